"""The FP64 operator on orthogonal meshes to the last digits that a solve needs.  Its rounding must not act
as a source: an error of eps rho(A) of one sign in every element, where rho(A) grows as n^2 K^4, comes back
from a solve as n^2 eps in the stream function, past any tolerance that the solve reports."""
import functools

import numpy as np
import pytest

import hoc
from hoc import meshes

pytestmark = pytest.mark.gpu

LD = np.longdouble


@functools.lru_cache(maxsize=None)
def tables(K):
    """Gauss points and weights, derivatives, end values and the Radau correction's derivative, in 80 bits."""
    P = np.polynomial.legendre
    c = np.zeros(K + 1, LD)
    c[K] = 1
    x = P.leggauss(K)[0].astype(LD)
    dc = P.legder(c)
    for _ in range(4):
        x = x - P.legval(x, c) / P.legval(x, dc)
    D, lv, ld = np.zeros((K, K), LD), np.zeros((K, 2), LD), np.zeros((K, 2), LD)

    def basis(m, s):  # value and derivative of the Lagrange polynomial m
        o = [q for q in range(K) if q != m]
        den = np.prod([x[m] - x[q] for q in o])
        v = np.prod([s - x[q] for q in o]) / den
        return v, sum(np.prod([s - x[q] for q in o if q != r], initial=LD(1)) for r in o) / den

    for m in range(K):
        for k in range(K):
            D[m, k] = basis(m, x[k])[1]
        for b, s in enumerate((LD(-1), LD(1))):
            lv[m, b], ld[m, b] = basis(m, s)
    r = np.zeros(K + 1, LD)  # (-1)^K (P_K - P_{K-1}) / 2
    r[K], r[K - 1] = LD((-1) ** K) / 2, -LD((-1) ** K) / 2
    dr = P.legder(r)
    return x, D, lv, ld, np.stack([P.legval(x, dr), -P.legval(-x, dr)], 1)


def second(u, K):
    """The FR line operator of -1 .. 1 cells with zero end values, on lines [.., cell, point]."""
    x, D, lv, ld, gd = tables(K)
    gp = np.array([-LD(K * (K + 1)) / 2, LD(K * (K + 1)) / 2])
    v, d = u @ lv, u @ ld
    cv = np.zeros_like(v)
    cv[..., :-1, 1] = cv[..., 1:, 0] = (v[..., :-1, 1] + v[..., 1:, 0]) / 2
    F = d + (cv - v) * gp
    F[..., :-1, 1] = F[..., 1:, 0] = (F[..., :-1, 1] + F[..., 1:, 0]) / 2
    q = u @ D + (cv - v) @ gd.T
    return q @ D + (F - q @ lv) @ gd.T


@pytest.mark.parametrize("precision", [hoc.HOC_FP64, hoc.HOC_MIXED])
@pytest.mark.parametrize("n,K", [(101, 6), (127, 5), (256, 5), (200, 4), (256, 3), (256, 2)])
def test_solve_of_known_solution(gpu_available, n, K, precision):
    x = tables(K)[0]
    s = ((np.arange(n)[:, None] + (1 + x)[None, :] / 2) / n).astype(LD)  # [cell, point]
    X, Y = s[None, None], s[:, :, None, None]                           # fields [row, j, column, i]
    psi = np.sin(LD(np.pi) * X) * Y * (1 - Y) * np.exp(X * Y) + np.sin(2 * LD(np.pi) * Y) * X * (1 - X) / 4
    A = second(psi, K) + np.moveaxis(second(np.moveaxis(psi, (0, 1), (2, 3)), K), (2, 3), (0, 1))
    flat = lambda f: np.ascontiguousarray(f.transpose(0, 2, 1, 3), dtype=np.float64).ravel()  # noqa: E731
    w = flat(-A * (4 * LD(n) * n))  # A psi + J omega = 0, J = 1 / (4 n^2)
    g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-4, tol=1e-14, maxiter=400, precision=precision)
    g.load_mesh(meshes.cavity(n, 2))
    g.setup()
    got, want = g.poisson(w), flat(psi)
    e = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("n", n, "K", K, "its", g.stats()["last_iters"], "rel", e)
    # the tolerance times ||A psi|| / (lambda_min ||psi||), under 10 here, and the rounding of n cells in a row
    # of K^2-fold sums, eps n K^2 = 8e-13 at 101 cells of K = 6
    assert e <= 1e-13 + np.finfo(float).eps * n * K * K
    g.close()

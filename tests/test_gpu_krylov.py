"""The Poisson iterations in every form their launches take: the iteration's test in a block of the next
smoothing step (small meshes, two or more steps) or in a launch of its own (one step, or more partial
sums than a block adds up); PCG and BiCGSTAB; FP64 and mixed precision; the coarse product with the
gather of its right-hand side at both of its sizes and past them.  The result is judged by the operator
itself, applied outside the solve: the cavity's stream function is zero on its walls, so A psi + J omega
(A: the Laplacian times the Jacobian J) is the residual."""
import numpy as np
import pytest

import hoc
from hoc import meshes

pytestmark = pytest.mark.gpu

TOL = 1e-8


def jacobian(g, K):
    """The Jacobian at the solution points, by differentiating their coordinates along the Gauss points."""
    xi = np.polynomial.legendre.leggauss(K)[0]
    d = np.array([[sum(np.prod([(xi[a] - xi[m]) / (xi[i] - xi[m]) for m in range(K) if m not in (i, q)]) / (xi[i] - xi[q])
                       for q in range(K) if q != i) for i in range(K)] for a in range(K)])
    p = g.solution_points().reshape(-1, K, K, 2)
    px, pe = np.einsum("ai,njic->njac", d, p), np.einsum("aj,njic->naic", d, p)
    return np.abs(px[..., 0] * pe[..., 1] - px[..., 1] * pe[..., 0]).ravel()


@pytest.mark.parametrize("precision", [hoc.HOC_FP64, hoc.HOC_MIXED])
@pytest.mark.parametrize("n,K,curved,cheb", [
    (16, 3, False, 0), (17, 3, False, 0),    # 289 and 324 vertices: the two register counts of the product
    (33, 2, False, 0), (34, 2, False, 0),    # 1156 vertices, and 1225: past the size of the fused product
    (6, 4, False, 1), (6, 4, True, 1),       # one smoothing step
    (9, 5, True, 3), (16, 2, True, 0),
    (203, 6, False, 0), (203, 6, True, 0),   # 1031 partial sums
])
def test_residual(gpu_available, n, K, curved, cheb, precision):
    m = meshes.cavity(n, 2, seed=n, jitter=0.1 if curved else 0.0)
    g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-4, tol=TOL, maxiter=400, precision=precision, cheb_degree=cheb)
    g.load_mesh(m)
    g.setup()
    w = np.random.default_rng(n).standard_normal(g.D)
    b = jacobian(g, K) * w
    for scale in (1.0, 0.0, 2.0):  # a second solve from the first one's state, with a zero one in between
        psi = g.poisson(scale * w)
        if scale == 0.0:
            assert not psi.any()
            continue
        e = np.linalg.norm(g.apply_laplacian(psi) + scale * b) / np.linalg.norm(scale * b)
        st = g.stats()
        print("n", n, "K", K, "curved", curved, "cheb", cheb, "its", st["last_iters"], "residual", e)
        # the rounding of A psi adds eps |A| |psi| / |omega| < 1e-11 here
        assert 0 < st["last_iters"] < 400 and e <= 1.01 * TOL
    g.close()


def test_iteration_budget(gpu_available):
    """maxiter stops the iterations at the same count in both forms of the test."""
    m = meshes.cavity(8, 2, seed=1, jitter=0.1)
    for cheb in (1, 2):
        g = hoc.HO2D(K=3, problem_type=1, Re=100.0, dt=1e-4, tol=1e-14, maxiter=3, cheb_degree=cheb)
        g.load_mesh(m)
        g.setup()
        g.poisson(np.random.default_rng(0).standard_normal(g.D))
        assert g.stats()["last_iters"] == 3
        g.close()

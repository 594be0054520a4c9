"""The smoother chosen by order and element shape, on both sides of each line between the choices: the
same iterates as with that degree and interval given, and a solution that the operator itself, applied
outside the solve, confirms (A psi + J omega is the residual, J the Jacobian)."""
import numpy as np
import pytest

import hoc
from hoc import meshes
from test_gpu_krylov import jacobian

pytestmark = pytest.mark.gpu

TOL = 1e-8


def solve(m, K, w, **options):
    g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-4, tol=TOL, maxiter=400, launch_mode=1, **options)
    g.load_mesh(m)
    g.setup()
    psi = g.poisson(w)
    e = np.linalg.norm(g.apply_laplacian(psi) + jacobian(g, K) * w) / np.linalg.norm(jacobian(g, K) * w)
    its = g.stats()["last_iters"]
    g.close()
    return psi, its, e


@pytest.mark.parametrize("jitter", [0.0, 0.1])
@pytest.mark.parametrize("K,ratio,degree,lower", [
    (2, 2.8, 2, 0.15), (2, 3.2, 3, 0.05), (3, 1.4, 2, 0.15), (3, 1.6, 3, 0.05), (4, 1.4, 2, 0.12),
    (5, 1.4, 2, 0.1), (5, 1.6, 3, 0.05), (6, 1.0, 3, 0.06), (6, 20.0, 4, 0.03),
    (2, 5.0, 3, 0.05), (3, 2.8, 3, 0.05), (3, 3.2, 4, 0.03), (4, 2.8, 3, 0.05), (4, 3.2, 4, 0.03), (5, 2.0, 4, 0.03),
    (6, 1.6, 3, 0.06), (6, 2.0, 4, 0.03),
])
def test_choice(gpu_available, K, ratio, degree, lower, jitter):
    m = meshes.cavity(11, 2, seed=3, jitter=jitter * min(1.0, 2.0 / ratio) if ratio < 10 else 0.0)
    m = meshes.QuadMesh(m.lnod, m.xy * np.array([1.0, 1.0 / ratio]), m.elem, m.bedges, m.bedge_bdry, m.bnames)
    w = np.random.default_rng(K).standard_normal(m.n_elem * K * K)
    psi, its, e = solve(m, K, w)
    same, its2, _ = solve(m, K, w, cheb_degree=degree, cheb_lower=lower)
    print("K", K, "ratio", ratio, "jitter", jitter, "its", its, "residual", e)
    assert its == its2 and np.array_equal(psi, same)
    # the rounding of A psi adds eps |A| |psi| / |omega| < 1e-11 here
    assert 0 < its < 400 and e <= 1.01 * TOL


def test_given_degree_keeps_its_interval(gpu_available):
    m = meshes.cavity(11, 2)
    w = np.random.default_rng(0).standard_normal(m.n_elem * 9)
    a, b = solve(m, 3, w, cheb_degree=3), solve(m, 3, w, cheb_degree=3, cheb_lower=0.1)
    assert a[1] == b[1] and np.array_equal(a[0], b[0])

"""Solves that end by a breakdown of the Krylov method.  With a zero tolerance the recursive residual shrinks
until r.z or p.q underflows, which ends the solve: x stays that of the iteration
before, the same from run to run, and a solve after it starts afresh."""
import numpy as np
import pytest

import hoc
from hoc import meshes
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,curved,cheb,launch_mode", [
    (9, 3, False, 0, 1), (33, 4, False, 0, 1), (33, 4, False, 0, 2),  # one and many blocks; replayed graphs
    (9, 3, False, 1, 1),                                             # the test in a launch of its own
    (12, 4, True, 0, 1),                                             # BiCGSTAB
])
def test_breakdown_keeps_the_solution(gpu_available, n, K, curved, cheb, launch_mode):
    m = meshes.cavity(n, 2, seed=n, jitter=0.1 if curved else 0.0)

    def handle(tol):
        g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-4, tol=tol, maxiter=3000,
                     cheb_degree=cheb, launch_mode=launch_mode, psi_guess=1)
        g.load_mesh(m)
        g.setup()
        return g

    g = handle(1e-13)
    w, w2 = np.random.default_rng(n).standard_normal((2, g.D))
    want, want2 = g.poisson(w), g.poisson(w2)
    g.close()
    g = handle(0.0)
    first = None
    for _ in range(8):
        g.set_streamfunction(np.zeros(g.D))
        psi = g.poisson(w)
        st = g.stats()
        assert 0 < st["last_iters"] < 3000
        # both solve to 1e-13 or below of a system whose condition number is below 1e5 at these sizes
        assert rel_l2(psi, want) < 1e-8
        if first is None:
            first = (psi, st["last_iters"])
            print("n", n, "K", K, "curved", curved, "cheb", cheb, "its", st["last_iters"], "residual",
                  st["last_rel_residual"])
        assert np.array_equal(psi, first[0]) and st["last_iters"] == first[1]
    assert rel_l2(g.poisson(w2), want2) < 1e-8
    g.close()

"""The adjoint's probes in batches of several colours: all units in one batch, an uneven last batch, and
few units a batch, against central differences of the stage map."""
import numpy as np
import pytest

import hoc
from hoc import meshes

pytestmark = pytest.mark.gpu


# units of the two maps (colours; twice the colours) and what a batch holds: all; 12; 3
@pytest.mark.parametrize("n,K", [(9, 5), (64, 3), (48, 5)])
def test_stage_vjp(gpu_available, n, K):
    g = hoc.HO2D(K=K, problem_type=1, Re=1000.0, dt=1e-3, time_integration_type=4, advection_type=1, tol=1e-14,
                 maxiter=800)
    g.load_mesh(meshes.cavity(n, 2))
    g.setup()
    rng = np.random.default_rng(n)
    e = np.arange(n * n)
    # jumps of 4 or more across every face: no flux point near the 1e-4 threshold of the upwind switch
    w = rng.uniform(-1, 1, g.D) + np.repeat(3.0 * (-1.0) ** (e // n + e % n), K * K)
    lam, v = rng.standard_normal(g.D), rng.standard_normal(g.D)
    gw, _ = g.stage_vjp(w, lam)
    eps = 1e-7
    fd = (g.stage(w + eps * v) - g.stage(w - eps * v)) / (2 * eps)
    lhs, rhs = gw @ v, lam @ fd
    print("n", n, "K", K, lhs, rhs, abs(lhs - rhs) / abs(rhs))
    # the solves' 1e-14 over eps, and 1e3 of room for the cancellation in the sums; a unit that is left
    # out or gathered twice is an error of order 1 / 14
    assert abs(lhs - rhs) <= 1e-4 * abs(rhs)
    g.close()

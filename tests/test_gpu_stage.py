"""The right-hand side, velocity and stage kernels (K lanes per element) at the edges of their wavefronts
and blocks, on every geometry they are instantiated for, with inflow, outflow and wall boundaries and
every pairing of neighbouring faces, both advection schemes: one stage against the FP64 oracle.  And
steps of the three time integrators, whose stages may not read what they write."""
import numpy as np
import pytest

import hoc
from hoc import meshes
from pyoracle import Oracle
from conftest import rel_l2
from test_gpu_fine import EPW, strip

pytestmark = pytest.mark.gpu


def handles(m, K, pt, integ, adv):
    c = dict(problem_type=pt, Re=100.0, dt=1e-4, time_integration_type=integ, advection_type=adv, tol=1e-14, maxiter=900)
    g = hoc.HO2D(K=K, **c)
    g.load_mesh(m)
    g.setup()
    return g, Oracle(m, K, **c)


@pytest.mark.parametrize("kind", ["ortho", "skewed", "point"])
@pytest.mark.parametrize("K", [2, 3, 4, 5, 6])
def test_stage_at_tile_edges(gpu_available, K, kind):
    rng = np.random.default_rng(K)
    for i, n in enumerate((1, EPW[K] - 1, EPW[K], EPW[K] + 1, 4 * EPW[K] - 1, 4 * EPW[K], 4 * EPW[K] + 1)):
        g, o = handles(strip(n, kind, seed=n), K, 2, 4, 1 + i % 2)
        w = rng.standard_normal(g.D)
        e = rel_l2(g.stage(w, 3.0), o.stage(w, 3.0))
        print(kind, "K", K, "elements", n, "advection", 1 + i % 2, "rel", e)
        # both solves to 1e-14 of a system whose condition number is below 1e7 on these strips
        assert e < 1e-7
        g.close()


@pytest.mark.parametrize("integ", [1, 2, 4])
@pytest.mark.parametrize("kind,adv", [("ortho", 1), ("ortho", 2), ("point", 1), ("point", 2)])
def test_steps(gpu_available, kind, adv, integ):
    m = meshes.backward_facing_step(24, 4, 2, jitter=0.1 if kind == "point" else 0.0, seed=3)
    g, o = handles(m, 4, 2, integ, adv)
    w = 0.1 * np.random.default_rng(adv).standard_normal(g.D)
    g.set_vorticity(w)
    o.set_vorticity(w)
    g.step(3)
    o.step(3)
    ew, ev = rel_l2(g.get_vorticity(), o.vorticity()), rel_l2(g.get_velocity().ravel(), np.ravel(o.velocity()))
    print(kind, "integrator", integ, "advection", adv, "vorticity", ew, "velocity", ev)
    assert ew < 1e-9 and ev < 1e-9
    g.close()

"""The fine-level Poisson kernels (K lanes per element, neighbour lines read from the field) at the
sizes where their mapping can go wrong: meshes of fewer elements than a wavefront holds, exact
multiples of a wavefront's and of a block's elements, one more and one less, every K, on the three
geometries they are instantiated for (constant orthogonal, constant skewed, per-point metrics), with
every pairing of neighbouring faces (randomly rotated element frames).  The operator and a solve are
compared with the FP64 oracle; solves also cover the smoother and the V-cycle's transfers."""
import numpy as np
import pytest

import hoc
from hoc import meshes
from pyoracle import Oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu

EPW = {2: 32, 3: 20, 4: 16, 5: 12, 6: 10}  # elements per wavefront


def strip(n_elem, kind, seed):
    """n_elem elements in a row of unit cells (rotated frames), or the nearest n x 2 block."""
    m = meshes.backward_facing_step(n_elem, 1, 2, length=float(n_elem), height=1.0, step_len=0.0, step_h=0.0,
                                    rotate=True, seed=seed)
    if kind == "skewed":
        m.xy[:, 0] += 0.3 * m.xy[:, 1]
    elif kind == "point":
        m.xy[:, 1] *= 1.0 + 0.2 * np.sin(m.xy[:, 0])
    return m


def handles(m, K, pt, **kw):
    c = dict(problem_type=pt, Re=100.0, dt=1e-4, time_integration_type=4, advection_type=1, tol=1e-13, maxiter=400)
    g = hoc.HO2D(K=K, **c, **kw)
    g.load_mesh(m)
    g.setup()
    return g, Oracle(m, K, **c)


@pytest.mark.parametrize("kind", ["ortho", "skewed", "point"])
@pytest.mark.parametrize("K", [2, 3, 4, 5, 6])
def test_apply_at_tile_edges(gpu_available, K, kind):
    rng = np.random.default_rng(K)
    for n in (1, EPW[K] - 1, EPW[K], EPW[K] + 1, 4 * EPW[K] - 1, 4 * EPW[K], 4 * EPW[K] + 1):
        g, o = handles(strip(n, kind, seed=n), K, 2)
        x = rng.standard_normal(g.D)
        e = rel_l2(g.apply_laplacian(x), o.laplacian_mf(x))
        print(kind, "K", K, "elements", n, "rel", e)
        # second differences of O(1) data: cancellation of at most the operator's largest entries, ~1e3 roundings
        assert e < 1e-12
        g.close()


@pytest.mark.parametrize("precision", [hoc.HOC_FP64, hoc.HOC_MIXED])
@pytest.mark.parametrize("K,n,kind", [(2, 9, "ortho"), (3, 7, "ortho"), (4, 5, "skewed"), (5, 7, "point"), (6, 7, "ortho"),
                                      (5, 11, "ortho")])
def test_solve_against_oracle(gpu_available, K, n, kind, precision):
    m = meshes.cavity(n, 2, seed=n, rotate=True, jitter=0.1 if kind == "point" else 0.0)
    if kind == "skewed":
        m.xy[:, 0] += 0.3 * m.xy[:, 1]
    g, o = handles(m, K, 1, precision=precision)
    w = np.random.default_rng(n).standard_normal(g.D)
    e = rel_l2(g.poisson(w), o.poisson(w))
    st = g.stats()
    print(kind, "K", K, "n", n, "rel", e, "its", st["last_iters"], "residual", st["last_rel_residual"])
    assert st["last_rel_residual"] <= 1e-13
    # both sides solve to 1e-13 of a system whose condition number is below ~1e4 at these sizes
    assert e < 1e-9
    g.close()

"""The Poisson operator applied through an ensemble's handle, after solves that left every instance
stopped (no operator launch of the handle's own behind them): the host and the device entry against the
same operator through a handle of each instance's own."""
import ctypes as C

import numpy as np
import pytest

import hoc
from hoc import meshes
from test_zz_no_alloc import DevBuf, _hip

pytestmark = pytest.mark.gpu

SIZES = (16, 30, 21)  # at 64 elements a block: several blocks inside each instance


def handle(m, K, precision, off=None, **kw):
    g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-5, tol=1e-12, maxiter=400, precision=precision, **kw)
    g.load_mesh(m)
    if off is not None:
        n = len(off) - 1
        g.set_instances(off, 100.0 * np.arange(1, n + 1), np.full(n, 1e-5))
    g.setup()
    return g


@pytest.mark.parametrize("precision", [hoc.HOC_FP64, hoc.HOC_MIXED])
@pytest.mark.parametrize("solve", ["poisson", "zero", "step"])
def test_apply_after_solve(gpu_available, solve, precision):
    K, rng = 4, np.random.default_rng(3)
    parts = [meshes.cavity(n, 2) for n in SIZES]
    m, off = meshes.concat(parts)
    g = handle(m, K, precision, off, psi_guess=4)  # no projection, whose append applies the operator
    x = rng.standard_normal(g.D)
    if solve == "poisson":
        g.poisson(rng.standard_normal(g.D))
    elif solve == "zero":
        g.poisson(np.zeros(g.D))
    else:
        g.step(1)
    hip = _hip()
    hip.hipDeviceSynchronize.argtypes = []
    xd, yd = DevBuf(hip, g.D), DevBuf(hip, g.D)
    xd.put(x)
    yd.put(np.full(g.D, np.nan))
    g.apply_laplacian_device(xd.p.value, yd.p.value, 0)
    assert hip.hipDeviceSynchronize() == 0
    y = {"device": yd.get(), "host": g.apply_laplacian(x)}
    xd.free(); yd.free()
    for i, part in enumerate(parts):
        sl = slice(off[i] * K * K, off[i + 1] * K * K)
        o = handle(part, K, hoc.HOC_FP64)
        want = o.apply_laplacian(x[sl])
        o.close()
        for entry, got in y.items():
            e = np.abs(got[sl] - want).max() / np.abs(want).max()
            print(solve, "instance", i, entry, "max relative difference", e)
            assert e <= 1e-15  # the same operations on the same values
    g.close()

"""Results of a few bytes to some tens of MB into the caller's memory: pageable memory (past 8 MB through a
ring of pinned chunks), pinned memory, which the device writes by itself, and an odd address inside either."""
import numpy as np
import pytest
import torch

import hoc
from hoc import meshes

pytestmark = pytest.mark.gpu


# 8 MiB hold 1048576 values: below, just above (a short ninth chunk), and 17 chunks and a bit (slots are reused)
@pytest.mark.parametrize("n,K", [(8, 3), (181, 5), (255, 4), (257, 4), (300, 5)])
def test_results_into_any_host_memory(gpu_available, n, K):
    g = hoc.HO2D(K=K, problem_type=1, Re=100.0, dt=1e-5, launch_mode=1)
    g.load_mesh(meshes.cavity(n, 2))
    g.setup()
    w = np.random.default_rng(n).standard_normal(g.D)
    g.set_vorticity(w)
    pinned = torch.empty(g.D + 3, dtype=torch.float64).pin_memory().numpy()
    for kind, buf in (("pageable", np.empty(g.D + 3)), ("pinned", pinned)):
        buf[:] = np.nan
        g._chk(hoc.lib().hoc_get_vorticity(g.h, g.D, buf[1:-2]))
        assert np.array_equal(buf[1:-2], w), kind
        assert np.isnan(buf[[0, -2, -1]]).all(), kind
    g.close()

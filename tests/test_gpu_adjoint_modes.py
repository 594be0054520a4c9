"""The adjoint's probe batches where not every unit fits one: the vorticity's units in one batch and the
velocity's in an uneven pair, several units a batch with an uneven last one, and one unit a batch."""
import pytest

from test_gpu_adjoint_batch import test_stage_vjp as stage_vjp

pytestmark = pytest.mark.gpu

COLOURS = 7  # of the distance-2 colouring of a grid: that many units of the vorticity, twice as many of U


def units_a_batch(n, K):
    """256 MiB over a unit's K^2 probes of 4 D + 4 N K values (adjoint_setup)."""
    N = n * n
    return max(1, int(2**28 / (8 * K * K * (4 * N * K * K + 4 * N * K))))


@pytest.mark.parametrize("n,K,units", [(80, 3, 12), (56, 5, 3), (64, 6, 1)])
def test_stage_vjp_in_batches(gpu_available, n, K, units):
    assert units_a_batch(n, K) == units < 2 * COLOURS
    stage_vjp(gpu_available, n, K)

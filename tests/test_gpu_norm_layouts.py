"""The norm of a call is the same bit for bit whichever kernel grids it: the
sums over the footprints do not depend on the layout of the tables (rows of
taps between zero rows, or padded to 8 or 16 taps)."""
import numpy as np
import pytest

from mi355_gridding import _lib
from test_gpu_bands import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("supports", [[0, 3, 7], [8, 31, 63]])
def test_norm_does_not_depend_on_the_kernel(gpu, supports):
    torch, ops = gpu
    c = _case(500, 4, supports, 3000, seed=4)
    # (53-bit taps: sums of 24-bit ones are exact in any order)
    c["conv_func"] = np.random.default_rng(5).normal(size=c["conv_func"].shape)
    grid0 = np.zeros((500, 500, 2))
    for dtype in (torch.float32, torch.float64):
        norms = [_run(torch, ops, c, dtype, grid0, **o)[1]
                 for o in ({}, dict(OPT_MIN_STAGE_RUN=3), dict(OPT_GRID_KERNEL=1),
                           dict(OPT_GRID_KERNEL=2), dict(OPT_COMPENSATED=1))]
        assert norms[0] != 0 and len(set(norms)) == 1, norms

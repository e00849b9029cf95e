"""Cell sums of the weighting pre-pass at the sizes where the sort's and the
sums' chunks end: cells that start in one chunk of sorted points and run on
over several, points off the grid behind them, and the index form that a
workspace cap selects in FP64.  Bar: the oracle's bits (the same additions in
the same order).
"""
import numpy as np
import pytest

from conftest import same_bits_or_nan
from oracle import oracle
from mi355_gridding import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", [np.float32, np.float64])
@pytest.mark.parametrize("n,long_cell,outside", [
    (1, 0, 0), (511, 400, 0), (512, 512, 0), (513, 513, 0), (1024, 512, 3),
    (4096, 3000, 7), (4097, 0, 4000), (20011, 1500, 100), (20011, 9000, 0),
])
@pytest.mark.parametrize("capped", [False, True])
def test_cell_sums(gpu, real, n, long_cell, outside, capped):
    torch, ops = gpu
    rng = np.random.default_rng(n + long_cell)
    G, cell = 128, real(1e-3)
    uv = (rng.integers(-40, 40, (2, n)) / (G * float(cell))).astype(real)
    uv[:, :long_cell] = real(3 / (G * float(cell)))
    uv[:, n - outside:] = real(900 / (G * float(cell)))
    uv = uv[:, rng.permutation(n)]
    weight = rng.lognormal(0, 3, n).astype(real)
    want = rng.standard_normal((G, G)).astype(real)
    grid = torch.from_numpy(want.copy()).cuda()
    skipped = oracle.weights_write(uv[0], uv[1], weight, cell, G, want)
    ctx = _lib.Context(torch.cuda.current_device())
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    if capped:
        ctx.set_option(_lib.OPT_MAX_WORKSPACE, 256 << 20)
    got = torch.full((1,), 99, dtype=torch.int64, device="cuda")
    u, v, w = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (uv[0], uv[1], weight))
    ops.grid_weights_write(u, v, w, float(cell), G, grid, got, ctx=ctx)
    torch.cuda.synchronize()
    ctx.close()
    assert int(got.item()) == skipped
    assert same_bits_or_nan(grid.cpu().numpy(), want)

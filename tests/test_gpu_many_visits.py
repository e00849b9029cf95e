"""FP64 calls of more than 2^30 tile visits (the 64 x 64 kernels take up to
2^32 - 1, so the band kernel does): 269 million visibilities whose 5 x 5
footprints straddle the corners of four regions, unit taps and amplitudes.
Every sum is a whole number below 2^53, so grid, norm and count are exact.

Needs about 110 GiB of device memory and a second.
"""
import numpy as np
import pytest

from mi355_gridding import _lib

pytestmark = pytest.mark.gpu

N = 269_000_003
G = 512


def test_more_than_2_to_30_visits_fp64(gpu):
    torch, ops = gpu
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("less than 160 GiB of device memory free")
    ks = ops.KernelStack([2], 1, 4, np.tile([1.0, 0.0], 16), dtype=torch.float64)
    # cells (128 a, 128 b), a and b in turn 1, 2, 3; one cell per wavelength
    i = torch.arange(N, device="cuda")
    uu = (G // 2 - 128.0 * (1 + i % 3)).double()
    vv = (128.0 * (1 + i // 3 % 3) - G // 2).double()
    count = torch.bincount(i % 9, minlength=9).view(3, 3).cpu().numpy()      # [b][a]
    del i
    ww = torch.zeros(N, dtype=torch.float64, device="cuda")
    weight = torch.ones(N, dtype=torch.float64, device="cuda")
    vis = torch.zeros((N, 2), dtype=torch.float64, device="cuda")
    vis[:, 0] = 1
    grid = torch.zeros((G, G, 2), dtype=torch.float64, device="cuda")
    norm = torch.zeros(1, dtype=torch.float64, device="cuda")
    sk = torch.zeros(1, dtype=torch.int64, device="cuda")
    ctx = _lib.Context(torch.cuda.current_device())
    try:
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ops.grid(ks, uu, vv, ww, vis, weight, 1.0 / G, 1.0, G, grid, norm, sk, ctx=ctx)
        torch.cuda.synchronize()
        assert ctx.stats()["num_visits"] == 4 * N > 1 << 30
    finally:
        ctx.close()
    del uu, vv, ww, vis, weight
    torch.cuda.empty_cache()
    want = np.zeros((G, G))
    for b in range(3):
        for a in range(3):
            want[128 * (b + 1) - 2:128 * (b + 1) + 3, 128 * (a + 1) - 2:128 * (a + 1) + 3] = count[b, a]
    g = grid.cpu().numpy()
    assert np.array_equal(g[..., 0], want) and not g[..., 1].any()
    assert norm.item() == 25 * N and sk.item() == 0

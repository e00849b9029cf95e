"""Which kernel an automatic pass takes: FP32, plain and compensated, on both
sides of each line of the rule; FP64 with and without a workspace cap; and on
the shapes that the band kernel is checked on.  The kernels split regions into
different items, so that of random data a pass equals one with the strip kernel
asked for (by a staging threshold that is the automatic one) bit for bit only
where it took that kernel."""
import numpy as np
import pytest

from mi355_gridding import _lib
from test_gpu_bands import SUPPORTS, _case, _run

pytestmark = pytest.mark.gpu

LARGE = 5888          # 23 x 46 regions of 256 x 128: more than 1024
SMALL = 5632          # 22 x 44: fewer


def _grid(torch, ops, c, comp, strips):
    ctx = _lib.Context(torch.cuda.current_device())
    try:
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ctx.set_option(_lib.OPT_COMPENSATED, comp)
        ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 6 if strips else 0)
        ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"], c["conv_func"])
        d = {k: torch.from_numpy(c[k]).cuda() for k in ("uu", "vv", "ww", "vis", "weight")}
        G = c["grid_size"]
        g = torch.zeros((G, G, 2), dtype=torch.float32, device="cuda")
        norm = torch.zeros(1, dtype=torch.float64, device="cuda")
        sk = torch.zeros(1, dtype=torch.int64, device="cuda")
        ops.grid(ks, d["uu"], d["vv"], d["ww"], d["vis"], d["weight"], c["cell_size_rad"],
                 c["w_scale"], G, g, norm, sk, ctx=ctx)
        torch.cuda.synchronize()
        return g
    finally:
        ctx.close()


# (compensated, grid, largest support, planes, oversampling, visibilities, bands?);
# oversampling 1: 4 tables a plane, 4: 9
@pytest.mark.parametrize("comp,G,smax,P,ov,N,bands", [
    (0, SMALL, 17, 1, 1, 84_000, True), (0, LARGE, 17, 1, 1, 84_000, False),
    (0, LARGE, 17, 1, 1, 80_000, True), (0, LARGE, 16, 1, 1, 84_000, True),
    (0, LARGE, 49, 8, 4, 999_999, True), (0, LARGE, 49, 8, 4, 1_000_000, False),
    (0, SMALL, 49, 8, 4, 1_000_000, True), (0, LARGE, 48, 8, 4, 1_000_000, True),
    (1, 700, 24, 1, 1, 65_532, True), (1, 700, 24, 1, 1, 65_536, False),
    (1, 700, 36, 2, 4, 53_999, True), (1, 700, 36, 2, 4, 54_000, False),
    (1, 700, 37, 2, 4, 17_999, True), (1, 700, 48, 2, 4, 18_000, False),
    (1, 700, 60, 3, 4, 399_999, True), (1, 700, 60, 3, 4, 400_000, False),
    (1, 700, 61, 3, 4, 149_999, True), (1, 700, 72, 3, 4, 150_000, False),
    (1, 900, 73, 3, 4, 2000, False), (1, 900, 72, 3, 4, 2000, True)])
def test_rule_of_the_automatic_choice(gpu, comp, G, smax, P, ov, N, bands):
    torch, ops = gpu
    supports = np.linspace(smax, max(1, smax - 8), P).astype(int).tolist()
    c = _case(G, ov, supports, N, seed=N % 97)
    assert max(supports) == smax and len(supports) == P
    auto = _grid(torch, ops, c, comp, False)
    strips = _grid(torch, ops, c, comp, True)
    assert torch.equal(auto, strips) != bands
    assert (auto - strips).abs().max() <= 1e-4 * strips.abs().max()


@pytest.mark.parametrize("G,ov,supports,n", [(333, 4, SUPPORTS, 3000), (640, 3, SUPPORTS, 2000),
                                             (130, 1, [0, 1, 2], 4000), (1030, 4, [70], 4000),
                                             (257, 8, [8, 9], 5000)])
def test_shapes_of_the_band_checks(gpu, G, ov, supports, n):
    """(Enough visibilities for several items a region: the kernels add one
    item's visits in the same order.)"""
    torch, ops = gpu
    c = _case(G, ov, supports, n, seed=G)
    grid0 = np.random.default_rng(1).normal(size=(G, G, 2))
    for dtype, opts, other in ((torch.float32, {}, dict(OPT_MIN_STAGE_RUN_W33=6)),
                               (torch.float32, dict(OPT_COMPENSATED=1),
                                dict(OPT_COMPENSATED=1, OPT_MIN_STAGE_RUN_W33=6)),
                               (torch.float64, {}, dict(OPT_GRID_KERNEL=2)),
                               (torch.float64, {}, dict(OPT_MAX_WORKSPACE=4 << 30))):
        a, an, _ = _run(torch, ops, c, dtype, grid0, **opts)
        b, bn, _ = _run(torch, ops, c, dtype, grid0, **other)
        assert not np.array_equal(a, b) and np.abs(a - b).max() <= 1e-5 * np.abs(b).max()
        assert an == bn


@pytest.mark.parametrize("points,smax,bands", [(333_333, 61, True), (333_334, 61, False),
                                               (333_334, 60, True)])
def test_rule_for_many_jobs_of_wide_footprints(gpu, points, smax, bands):
    """9 jobs on large grids: 3 million visibilities in all are the line for
    supports above 60, below that of each job (1 million)."""
    torch, ops = gpu
    c = _case(LARGE, 4, [smax, 3], points, seed=8)
    ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"], c["conv_func"])
    d = {k: torch.from_numpy(c[k]).cuda() for k in ("uu", "vv", "ww", "vis", "weight")}
    cat = {k: torch.cat([v] * 9) for k, v in d.items()}
    norm = torch.zeros(9, dtype=torch.float64, device="cuda")
    sk = torch.zeros(9, dtype=torch.int64, device="cuda")
    grids = []
    for strips in (False, True):
        g = torch.zeros((9, LARGE, LARGE, 2), dtype=torch.float32, device="cuda")
        jobs = [dict(vis_offset=j * points, num_points=points, cell_size_rad=c["cell_size_rad"],
                     w_scale=c["w_scale"], grid_size=LARGE, grid=g[j], norm=norm[j:j + 1],
                     num_skipped=sk[j:j + 1]) for j in range(9)]
        ctx = _lib.Context(torch.cuda.current_device())
        try:
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 6 if strips else 0)
            ops.grid_batched(ks, jobs, cat["uu"], cat["vv"], cat["ww"], cat["vis"], cat["weight"],
                             ctx=ctx)
            torch.cuda.synchronize()
        finally:
            ctx.close()
        grids.append(g)
    assert torch.equal(grids[0], grids[1]) != bands
    assert (grids[0] - grids[1]).abs().max() <= 1e-4 * grids[1].abs().max()

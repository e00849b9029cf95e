"""The band kernel (the automatic choice for FP64, and for FP32 and
compensated FP32 where tables serve few visits) against the serial oracle:
tables of every width class its units make (one column to ten units, widths
just below, at and above a unit's 8 or 16 columns), all four mirror
orientations, both conjugations, footprints across block (64 / 128 columns),
band (8 rows) and region borders, grids that end inside a block, several
items per region, odd oversampling, accumulation onto a non-zero grid.

Bars (norm-wise max error over max value): FP32 1e-5 (and the strip kernel's
grid of the same call within 1e-5), compensated 1e-6, FP64 1e-12;
num_skipped exact, norm 1e-12.  FP32 sums of at most a few thousand terms per
cell carry an error of a few 1e-7 of the largest cell.
"""
import numpy as np
import pytest

from conftest import errors
from oracle import oracle
from mi355_gridding import _lib

pytestmark = pytest.mark.gpu

SUPPORTS = [0, 1, 3, 4, 7, 8, 15, 16, 23, 31, 32, 39, 63, 64, 70]


def _case(G, ov, supports, n, seed):
    rng = np.random.default_rng(seed)
    P = len(supports)
    csh = ov * max(supports) + (ov + 1) // 2 + 1
    cell = np.float32(1.0 / G)                       # a cell per wavelength
    plane = rng.integers(0, P, n)
    ww = (plane.astype(np.float64) ** 2 * rng.choice([-1.0, 1.0], n)).astype(np.float32)
    span = 0.52 * G                                  # a few footprints leave the grid
    return dict(num_w_planes=P, support=np.array(supports, np.int32), oversample=ov,
                conv_size_half=csh,
                conv_func=rng.normal(size=(P, csh, csh, 2)).astype(np.float32), num_points=n,
                uu=rng.uniform(-span, span, n).astype(np.float32),
                vv=rng.uniform(-span, span, n).astype(np.float32), ww=ww,
                vis=rng.normal(size=(n, 2)).astype(np.float32),
                weight=rng.uniform(0.5, 1.5, n).astype(np.float32), cell_size_rad=cell,
                w_scale=np.float32(1.0), grid_size=G)


def _run(torch, ops, c, dtype, grid0, **opts):
    ctx = _lib.Context(torch.cuda.current_device())
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    try:
        for k, v in opts.items():
            ctx.set_option(getattr(_lib, k), v)
        ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"], c["conv_func"],
                             dtype=dtype)
        d = {k: torch.from_numpy(c[k]).cuda().to(dtype).contiguous()
             for k in ("uu", "vv", "ww", "vis", "weight")}
        g = torch.from_numpy(grid0).cuda().to(dtype)
        norm = torch.zeros(1, dtype=torch.float64, device="cuda")
        sk = torch.zeros(1, dtype=torch.int64, device="cuda")
        ops.grid(ks, d["uu"], d["vv"], d["ww"], d["vis"], d["weight"], c["cell_size_rad"],
                 c["w_scale"], c["grid_size"], g, norm, sk, ctx=ctx)
        torch.cuda.synchronize()
        return g.cpu().numpy().astype(np.float64), norm.item(), int(sk.item())
    finally:
        ctx.close()


@pytest.mark.parametrize("G,ov,supports,n,vpi", [
    (333, 4, SUPPORTS, 3000, 0),            # odd grid, regions cut off on both sides
    (640, 3, SUPPORTS, 2000, 0),            # odd oversampling, off = +-2 of 3
    (130, 1, [0, 1, 2], 4000, 0),           # one table per plane, two blocks and a bit
    (1030, 4, [70], 400, 16),               # widest only, many items per region
    (257, 8, [8, 9], 5000, 0),              # tables one column past a unit
])
def test_band_kernel_against_oracle(gpu, G, ov, supports, n, vpi):
    torch, ops = gpu
    c = _case(G, ov, supports, n, seed=G)
    rng = np.random.default_rng(1)
    grid0 = rng.normal(size=(G, G, 2)).astype(np.float32).astype(np.float64)
    opts = dict(OPT_VISITS_PER_ITEM=vpi) if vpi else {}
    t, tn, ts = oracle.grid_fsel_d(c, grid=grid0.copy(), norm=0.0)
    g, nn, s = _run(torch, ops, c, torch.float32, grid0, **opts)
    assert s == ts and 0 < s < n and abs(nn - tn) <= 1e-12 * abs(tn)
    assert errors(g, t)[0] <= 1e-5
    strips, _, _ = _run(torch, ops, c, torch.float32, grid0, OPT_MIN_STAGE_RUN=3)
    assert errors(g, strips)[0] <= 1e-5
    comp, nn, s = _run(torch, ops, c, torch.float32, grid0, OPT_COMPENSATED=1, **opts)
    assert s == ts and errors(comp, t)[0] <= 1e-6
    t, tn, ts = oracle.grid_d(c, grid=grid0.copy(), norm=0.0)
    g, nn, s = _run(torch, ops, c, torch.float64, grid0, **opts)
    assert s == ts and abs(nn - tn) <= 1e-12 * abs(tn)
    assert errors(g, t)[0] <= 1e-12

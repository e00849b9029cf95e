"""The degridding kernel's units (8 rows x 8 lanes of two FP32 values or one
FP64 value): footprints one value wide up to several blocks of units, widths
just below, at and above a unit, all mirror orientations and conjugations,
footprints that end at the grid's last cell; and cells outside a footprint,
which may hold anything, never reach its sum.

Bars (norm-wise max error over max value, against the serial FP64 oracle with
the same selection): FP32 1e-5, FP64 1e-12.
"""
import numpy as np
import pytest

from conftest import errors
from oracle import oracle

pytestmark = pytest.mark.gpu

SUPPORTS = [0, 1, 3, 4, 7, 8, 11, 12, 15, 16, 31, 32, 63, 64, 70, 100]
G, OV = 512, 4


def _case(n, seed, supports=SUPPORTS):
    """Coordinates a safe distance from every rounding edge, so that FP32 and
    FP64 select the same cells and kernels (cell size 1/G: a cell per
    wavelength, exactly)."""
    rng = np.random.default_rng(seed)
    P = len(supports)
    plane = rng.integers(0, P, n)
    s = np.array(supports)[plane]
    cu, cv = (rng.integers(s, G - s) - G // 2 for _ in range(2))
    cu[:P], plane[:P] = G // 2 - 1 - np.array(supports), np.arange(P)   # to the last column
    cv[:P] = np.array([rng.integers(q, G - q) - G // 2 for q in supports])
    fu, fv = (0.25 * rng.integers(-1, 2, n) + 0.03 for _ in range(2))
    csh = OV * max(supports) + (OV + 1) // 2 + 1
    return dict(num_w_planes=P, support=np.array(supports, np.int32), oversample=OV,
                conv_size_half=csh,
                conv_func=rng.normal(size=(P, csh, csh, 2)).astype(np.float32), num_points=n,
                uu=-(cu - fu).astype(np.float32), vv=(cv - fv).astype(np.float32),
                ww=(plane.astype(np.float64) ** 2 * rng.choice([-1.0, 1.0], n)).astype(np.float32),
                vis=np.zeros((n, 2), np.float32),
                weight=rng.uniform(0.5, 1.5, n).astype(np.float32),
                cell_size_rad=np.float32(1.0 / G), w_scale=np.float32(1.0), grid_size=G)


def _degrid(torch, ops, c, grid, dtype):
    ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"], c["conv_func"],
                         dtype=dtype)
    d = [torch.from_numpy(c[k]).cuda().to(dtype) for k in ("uu", "vv", "ww", "weight")]
    out = ops.degrid(ks, *d, c["cell_size_rad"], c["w_scale"], G,
                     torch.from_numpy(grid).cuda().to(dtype))
    torch.cuda.synchronize()
    return out.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("n", [300, 5000])          # in index order, and in tile order
def test_degrid_units_against_oracle(gpu, n):
    torch, ops = gpu
    c = _case(n, seed=n)
    grid = np.random.default_rng(2).normal(size=(G, G, 2)).astype(np.float32)
    want = oracle.degrid_fsel_d(c, grid.astype(np.float64))
    assert errors(_degrid(torch, ops, c, grid, torch.float32), want)[0] <= 1e-5
    assert errors(_degrid(torch, ops, c, grid, torch.float64), want)[0] <= 1e-12


@pytest.mark.parametrize("support", [0, 3, 7, 8, 16, 63])
def test_degrid_reads_its_footprint_only(gpu, support):
    torch, ops = gpu
    for seed in range(4):
        c = _case(1, seed, [support])
        sel = oracle.select_f(c)
        x, y = int(sel["grid_u"][0]), int(sel["grid_v"][0])
        box = (slice(y - support, y + support + 1), slice(x - support, x + support + 1))
        clean = np.zeros((G, G, 2), np.float32)
        clean[box] = np.random.default_rng(seed).normal(size=clean[box].shape)
        grid = np.full((G, G, 2), np.nan, np.float32)
        grid[box] = clean[box]
        want = oracle.degrid_fsel_d(c, clean.astype(np.float64))
        assert errors(_degrid(torch, ops, c, grid, torch.float32), want)[0] <= 1e-5
        assert errors(_degrid(torch, ops, c, grid, torch.float64), want)[0] <= 1e-12

"""The degridding kernel that walks footprints flat, on the calls that take it:
large calls of small FP32 footprints, of wide FP32 ones with large tables, and
FP64 calls by size and support, one visibility above each line of the rule.
Against the serial FP64 oracle; against the other kernel, which a part of the
same visibilities takes (their sums agree to rounding, not bit for bit, which
tells the two apart); and with anything in the cells outside the footprint.

Bars as for the other kernel: FP32 1e-5, FP64 1e-12.
"""
import numpy as np
import pytest

from conftest import errors
from oracle import oracle
from test_gpu_degrid_units import G, _case, _degrid

pytestmark = pytest.mark.gpu

PART = 1000


@pytest.mark.parametrize("double,supports,n", [
    (False, [0, 1, 3, 4, 7, 8, 11], 100_001), (False, [11, 18], 100_000),
    (False, [57, 64] + [100] * 7, 4001),
    (True, [0, 1, 3, 4, 7, 8, 15, 16], 100_001), (True, [0, 3, 48], 30_000), (True, [32, 70], 2000)])
def test_flat_against_oracle_and_units(gpu, double, supports, n):
    torch, ops = gpu
    c = _case(n, seed=n, supports=supports)
    grid = np.random.default_rng(2).normal(size=(G, G, 2)).astype(np.float32)
    dtype, bar = (torch.float64, 1e-12) if double else (torch.float32, 1e-5)
    got = _degrid(torch, ops, c, grid, dtype)
    part = dict(c, num_points=PART, **{k: c[k][:PART] for k in ("uu", "vv", "ww", "vis", "weight")})
    want = oracle.degrid_fsel_d(part, grid.astype(np.float64))
    assert errors(got[:PART], want)[0] <= bar
    units = _degrid(torch, ops, part, grid, dtype)
    assert not np.array_equal(got[:PART], units) and errors(got[:PART], units)[0] <= bar
    last = dict(c, num_points=PART, **{k: c[k][-PART:] for k in ("uu", "vv", "ww", "vis", "weight")})
    assert errors(got[-PART:], oracle.degrid_fsel_d(last, grid.astype(np.float64)))[0] <= bar


@pytest.mark.parametrize("support", [0, 3, 4, 7, 11])
def test_flat_reads_its_footprint_only(gpu, support):
    torch, ops = gpu
    c = _case(1, 5, [support])
    sel = oracle.select_f(c)
    x, y = int(sel["grid_u"][0]), int(sel["grid_v"][0])
    box = (slice(y - support, y + support + 1), slice(x - support, x + support + 1))
    clean = np.zeros((G, G, 2), np.float32)
    clean[box] = np.random.default_rng(support).normal(size=clean[box].shape)
    grid = np.full((G, G, 2), np.nan, np.float32)
    grid[box] = clean[box]
    want = oracle.degrid_fsel_d(c, clean.astype(np.float64))
    n = 100_003
    many = dict(c, num_points=n, **{k: np.repeat(c[k], n, axis=0)
                                    for k in ("uu", "vv", "ww", "vis", "weight")})
    for dtype, bar in ((torch.float32, 1e-5), (torch.float64, 1e-12)):
        got = _degrid(torch, ops, many, grid, dtype)
        assert (got == got[0]).all() and errors(got[:1], want)[0] <= bar

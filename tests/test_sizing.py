"""The library's host arithmetic for buffer sizes and offsets
(csrc/gg_sizing.hpp), built here with the host compiler and called through
ctypes: no GPU, and sizes that no test could allocate."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

SHIM = r"""
#include "gg_sizing.hpp"
extern "C" size_t place(const int* sizes, int n, size_t* offsets)
{
    std::vector<size_t> o;
    const size_t cells = gg::place_grids(std::vector<int>(sizes, sizes + n), o);
    for (int i = 0; i < n; ++i) offsets[i] = o[i];
    return cells;
}
extern "C" unsigned long long slots(unsigned long long c, unsigned long long tiles,
        unsigned long long V)
{
    return gg::slot_bound(c, tiles, V);
}
extern "C" void item_sizes(const unsigned long long* points, const unsigned long long* tiles, int n,
        unsigned long long per_point, unsigned long long slot_bytes, unsigned coarsest,
        unsigned* sizes)
{
    std::vector<gg::JobSize> jobs;
    for (int i = 0; i < n; ++i) jobs.push_back({points[i], tiles[i]});
    std::vector<unsigned> out;
    gg::band_item_sizes(jobs, per_point, slot_bytes, coarsest, out);
    for (int i = 0; i < n; ++i) sizes[i] = out[i];
}
extern "C" unsigned long long budget() { return gg::kSlotBudget; }
"""


@pytest.fixture(scope="module")
def sizing(tmp_path_factory):
    d = tmp_path_factory.mktemp("sizing")
    (d / "shim.cpp").write_text(SHIM)
    so = str(d / "shim.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall", "-Werror",
                    "-I", os.path.join(PKG, "csrc"), str(d / "shim.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.place.restype = ctypes.c_size_t
    lib.slots.restype = lib.budget.restype = ctypes.c_ulonglong
    lib.slots.argtypes = [ctypes.c_ulonglong] * 3
    return lib


@pytest.mark.parametrize("sizes", [[4096] * 200, [8192] * 40, [16384] * 12, [1 << 20] * 3,
                                   [1, 65536, 333, 46341, 2, 1 << 20]])
def test_trial_grids_do_not_overlap(sizing, sizes):
    """Past 2^31 cells every offset still lies behind the grids before it and
    each grid inside the allocation."""
    n = len(sizes)
    offsets = (ctypes.c_size_t * n)()
    cells = sizing.place((ctypes.c_int * n)(*sizes), n, offsets)
    ends = np.cumsum([g * g for g in sizes], dtype=object)
    assert cells == ends[-1] and cells > 1 << 31
    assert list(offsets) == [0] + list(ends[:-1])


@pytest.mark.parametrize("V", [1, 7, 64, 1024])
def test_slot_bound_covers_every_split(sizing, V):
    """Random and worst splits of c visits over the tiles of a job: the partial
    regions of the tiles with two or more items stay within the bound, and one
    split reaches it (V above the number of tiles)."""
    rng = np.random.default_rng(V)
    for _ in range(300):
        tiles = int(rng.integers(1, 40))
        c = int(rng.integers(0, 60 * V + 2))
        bound = sizing.slots(c, tiles, V)
        for cut in (np.sort(rng.integers(0, c + 1, tiles - 1)),            # any
                    np.minimum(np.arange(1, tiles) * (V + 1), c),           # V + 1 each
                    np.minimum(np.arange(1, tiles) * (2 * V + 1), c)):
            visits = np.diff(np.r_[0, cut, c])
            items = -(-visits // V)
            assert items[items >= 2].sum() <= bound, (visits, V)
    for tiles in (1, 5):                            # tiles - 1 of V + 1, the rest in one
        c = (tiles - 1) * (V + 1) + 9 * V + 1
        if V > tiles:
            assert sizing.slots(c, tiles, V) == 2 * (tiles - 1) + 10


def _sizes(sizing, points, tiles, per_point, slot_bytes, coarsest):
    n = len(points)
    u64, out = ctypes.c_ulonglong, (ctypes.c_uint * n)()
    sizing.item_sizes((u64 * n)(*points), (u64 * n)(*tiles), n, u64(per_point), u64(slot_bytes),
                      ctypes.c_uint(coarsest), out)
    return list(out)


def _slots(sizing, points, tiles, per_point, sizes):
    return sum(sizing.slots(p * per_point, t, v) for p, t, v in zip(points, tiles, sizes))


def _coarsest(n, num_cu=256):
    v = 8192
    while v > 1024 and n < 6 * v * num_cu:
        v //= 2
    return v


# jobs, visibilities of each, grid size (supports below 64: four regions of
# 256 x 128 cells at most); partial regions of 256 KiB
@pytest.mark.parametrize("jobs,points,G", [
    (64, 600_000, 4096), (256, 600_000, 4096), (1000, 8192, 1024), (2000, 8192, 1024),
    (5000, 2000, 512), (1500, 2000, 512), (20_000, 500, 256), (1, 31_400_000, 16384),
    (8, 4_000_000, 8192), (1, 400_000_000, 16384), (24, 550_000, 4096)])
def test_partial_regions_of_a_captured_batch(sizing, jobs, points, G):
    """Within the budget, or, where even the coarse items of the other kernels
    are not, no more than those need."""
    slot = 256 << 10
    tiles = -(-G // 256) * -(-G // 128)
    coarsest = _coarsest(jobs * points)
    sizes = _sizes(sizing, [points] * jobs, [tiles] * jobs, 4, slot, coarsest)
    need = _slots(sizing, [points] * jobs, [tiles] * jobs, 4, sizes) * slot
    other = _slots(sizing, [points] * jobs, [tiles] * jobs, 4, [coarsest] * jobs) * slot
    assert need <= max(sizing.budget(), other)
    assert min(sizes) >= 64 and len(set(sizes)) == 1


def test_few_jobs_are_split_as_calls_of_their_own(sizing):
    points = [2000, 40_000, 66_000, 600_000, 3, 2_000_000, 17_000, 9000]
    tiles = [8 * i + 1 for i in range(8)]
    own = [_sizes(sizing, [p], [t], 4, 256 << 10, _coarsest(p))[0] for p, t in zip(points, tiles)]
    assert _sizes(sizing, points, tiles, 4, 256 << 10, _coarsest(sum(points))) == own
    many = _sizes(sizing, points * 2, tiles * 2, 4, 256 << 10, _coarsest(2 * sum(points)))
    assert many == [1024] * 16

"""What mi355_ctx_get_buckets reports after a band-kernel pass: the lists of
that pass whatever ran since without touching them, with shortened kernel
table ids too, and nothing where the header promises nothing."""
import ctypes

import numpy as np
import pytest

from oracle import oracle
from mi355_gridding import _lib, synth
from test_gpu_buckets import restate

pytestmark = pytest.mark.gpu


def _grid(torch, ops, c, ctx):
    G = c["grid_size"]
    ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"], c["conv_func"])
    d = {k: torch.from_numpy(np.ascontiguousarray(c[k])).cuda()
         for k in ("uu", "vv", "ww", "vis", "weight")}
    grid = torch.zeros((G, G, 2), dtype=torch.float32, device="cuda")
    norm = torch.zeros(1, dtype=torch.float64, device="cuda")
    sk = torch.zeros(1, dtype=torch.int64, device="cuda")
    ops.grid(ks, d["uu"], d["vv"], d["ww"], d["vis"], d["weight"], c["cell_size_rad"],
             c["w_scale"], G, grid, norm, sk, ctx=ctx)
    return ks, d, grid


def _buckets(ctx):
    lib = _lib.load()
    n, bits = ctypes.c_ulonglong(0), ctypes.c_int(0)
    _lib.check(lib.mi355_ctx_get_buckets(ctx.handle, ctypes.byref(n), ctypes.byref(bits), None,
                                         None, None, 0))
    keys, vis = np.zeros(n.value, np.uint32), np.zeros(n.value, np.uint32)
    flags = np.zeros(n.value, np.int32)
    p = lambda a: ctypes.c_void_p(a.ctypes.data)
    _lib.check(lib.mi355_ctx_get_buckets(ctx.handle, ctypes.byref(n), ctypes.byref(bits),
                                         p(keys), p(vis), p(flags), n.value))
    return keys, vis, flags, bits.value


def _context(torch):
    ctx = _lib.Context(torch.cuda.current_device())
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return ctx


def test_lists_survive_a_small_degridding(gpu):
    """4000 planes, 36000 tables: a key stands for two tables, so that the runs
    come from the records.  Against the restatement (no shortened ids), re-keyed;
    and the same again after a degridding call of 100 other visibilities, which
    rewrites the selection records but none of the lists."""
    torch, ops = gpu
    c = synth.make(2, num_points=20_000, grid_size=512, num_w_planes=4000, max_support=8, seed=5)
    key, vis, _, bits = restate(c, (1, 1, 1, 1))
    assert bits == 16
    table, region = key & 0xFFFF, key >> 16
    # (stable by region and table, so a stable sort by the shorter key of the
    # visits in their first order gives the library's)
    first = np.lexsort((vis, region))
    short = (region.astype(np.uint64) << 15 | table >> 1).astype(np.uint32)
    order = first[np.argsort(short[first], kind="stable")]
    key, vis, table = short[order], vis[order], table[order]
    start = np.r_[True, (key[1:] != key[:-1]) | (table[1:] != table[:-1])]
    run = np.cumsum(start) - 1
    staged = np.bincount(run)[run] >= 6             # (tables at most 33 wide)
    flags = staged.astype(np.int32) | (start.astype(np.int32) << 1)
    assert 0 < staged.sum() < len(staged)
    ctx = _context(torch)
    try:
        ks, d, grid = _grid(torch, ops, c, ctx)
        for again in (False, True):
            k, v, f, b = _buckets(ctx)
            assert b == 15
            assert np.array_equal(k, key) and np.array_equal(v, vis)
            assert np.array_equal(f, flags), again
            sub = {n: d[n][-100:].contiguous() for n in ("uu", "vv", "ww", "weight")}
            ops.degrid(ks, sub["uu"], sub["vv"], sub["ww"], sub["weight"], c["cell_size_rad"],
                       c["w_scale"], c["grid_size"], grid, ctx=ctx)
            torch.cuda.synchronize()
    finally:
        ctx.close()


def test_no_lists_of_compensated_bands(gpu):
    """Compensated bands have regions of 128 x 128 cells: no lists, where keys
    numbered over 256 x 128 regions are expected."""
    torch, ops = gpu
    c = synth.make(0, num_points=20_000, grid_size=1024, num_w_planes=64, max_support=16, seed=6)
    ctx = _context(torch)
    try:
        _grid(torch, ops, c, ctx)
        assert len(_buckets(ctx)[0]) > 0
        ctx.set_option(_lib.OPT_COMPENSATED, 1)
        _grid(torch, ops, c, ctx)
        with pytest.raises(_lib.GridderError) as e:
            _buckets(ctx)
        assert e.value.status == _lib.ERR_INVALID_ARG
    finally:
        ctx.close()

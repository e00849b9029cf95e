"""How the band kernel's passes are split into work items where their own item
sizes cannot be had: a workspace cap, the static scratch of the allocation-free
entry, a device without the memory.  All then take the size of the other
kernels, so that grids equal those with that size asked for bit for bit, call
after call and replay after replay.
"""
import ctypes

import numpy as np
import pytest

from conftest import same_bits
from mi355_gridding import _lib, synth
from test_gpu_batched import _snap, _zero
from test_zz_no_alloc import _call

pytestmark = pytest.mark.gpu


def _context(torch, **opts):
    ctx = _lib.Context(torch.cuda.current_device())
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    for k, v in opts.items():
        ctx.set_option(getattr(_lib, k), v)
    return ctx


def _jobs(torch, ops, num_jobs, points, G, P, smax):
    b = synth.make_batched(counts=[points] * min(num_jobs, 4), grid_size=G, num_w_planes=P,
                           max_support=smax)
    ks = ops.KernelStack(b["support"], b["oversample"], b["conv_size_half"], b["conv_func"])
    four = {k: torch.from_numpy(np.concatenate([j[k] for j in b["jobs"]])).cuda()
            for k in ("uu", "vv", "ww", "vis", "weight")}
    n = num_jobs * points
    d = {k: torch.cat([v] * -(-n // len(v)))[:n].contiguous() for k, v in four.items()}
    norm = torch.zeros(num_jobs, dtype=torch.float64, device="cuda")
    sk = torch.zeros(num_jobs, dtype=torch.int64, device="cuda")
    jobs = [dict(vis_offset=i * points, num_points=points,
                 cell_size_rad=b["jobs"][0]["cell_size_rad"], w_scale=b["jobs"][0]["w_scale"],
                 grid_size=G, grid=torch.zeros((G, G, 2), dtype=torch.float32, device="cuda"),
                 norm=norm[i:i + 1], num_skipped=sk[i:i + 1]) for i in range(num_jobs)]
    return ks, jobs, d["uu"], d["vv"], d["ww"], d["vis"], d["weight"]


def _run(torch, fn, args, ctx):
    _zero(args[1])
    fn(*args, ctx=ctx)
    torch.cuda.synchronize()
    return _snap(args[1]), ctx.stats()["num_items"]


def _equal(a, b):
    return all(same_bits(g0, g1) and n0 == n1 and s0 == s1
               for (g0, n0, s0), (g1, n1, s1) in zip(a, b))


@pytest.mark.parametrize("graph", [False, True])
def test_split_under_a_cap_does_not_depend_on_the_past(gpu, graph):
    """A cap that the call fits with room to spare, also once a larger call has
    gone before, and one that holds little more than the call needs: the same
    split every time."""
    torch, ops = gpu
    args = _jobs(torch, ops, 3, 20_000, 1024, 64, 16)
    larger = _jobs(torch, ops, 3, 60_000, 1024, 64, 16)
    fn = ops.grid_batched_graph if graph else ops.grid_batched
    ctx = _context(torch, OPT_VISITS_PER_ITEM=1024)
    want, items = _run(torch, fn, args, ctx)
    ctx.close()
    ctx = _context(torch)
    assert _run(torch, fn, args, ctx)[1] > items           # (its own sizes are smaller)
    ctx.close()
    for cap, calls in ((1 << 30, (args, args, larger, args)), (128 << 20, (args,) * 3)):
        ctx = _context(torch, OPT_MAX_WORKSPACE=cap)
        try:
            for call in calls:
                got, n = _run(torch, fn, call, ctx)
                assert call is larger or (n == items and _equal(got, want)), cap
        finally:
            ctx.close()


def test_static_scratch_takes_the_coarser_split(gpu):
    """100,000 visibilities: partial regions of 512 visits each would need more
    than the 64 MiB, those of 1024 do not."""
    torch, ops = gpu
    lib = _lib.load()
    c = synth.make(0, num_points=100_000, grid_size=1024, num_w_planes=48, max_support=14, seed=31)
    sup = np.ascontiguousarray(c["support"], np.int32)
    conv = torch.from_numpy(np.ascontiguousarray(c["conv_func"])).cuda()
    ctx = _context(torch)
    try:
        own = _call(torch, lib.mi355_grid_wproj_f_dev, ctx, c, sup, conv)
        own_items = ctx.stats()["num_items"]
        ctx.set_option(_lib.OPT_VISITS_PER_ITEM, 1024)
        want = _call(torch, lib.mi355_grid_wproj_f_dev, ctx, c, sup, conv)
        items = ctx.stats()["num_items"]
        ctx.set_option(_lib.OPT_VISITS_PER_ITEM, 0)
        assert own[0] == want[0] == 0 and items < own_items
        got = _call(torch, lib.mi355_grid_wproj_f_dev_noalloc, ctx, c, sup, conv)
        assert got[0] == 0 and ctx.stats()["num_items"] == items
        assert same_bits(got[1], want[1]) and got[2:] == want[2:]
    finally:
        ctx.close()


@pytest.mark.parametrize("graph", [False, True])
def test_device_without_the_memory_takes_the_coarser_split(gpu, graph):
    """12 captured jobs of 600,000 visibilities allow for 7 GiB of partial
    regions with items of 1024 visits, 2 GiB with 4096: on a device with 7 GiB
    left the pass runs, split as with 4096, and its replays with it.  (Eager,
    the counts are exact, and the same memory holds its own split.)"""
    torch, ops = gpu
    args = _jobs(torch, ops, 12, 600_000, 1024, 64, 16)
    fn = ops.grid_batched_graph if graph else ops.grid_batched
    ctx = _context(torch)
    own, own_items = _run(torch, fn, args, ctx)
    ctx.set_option(_lib.OPT_VISITS_PER_ITEM, 4096)
    want, items = _run(torch, fn, args, ctx)
    ctx.close()
    assert items < own_items
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hold = torch.empty(torch.cuda.mem_get_info()[0] - (7 << 30), dtype=torch.uint8, device="cuda")
    ctx = _context(torch)
    try:
        for rep in range(4):
            got, n = _run(torch, fn, args, ctx)
            if graph:
                assert n == items and _equal(got, want), rep
            else:
                assert n == own_items and _equal(got, own), rep
    finally:
        ctx.close()
        del hold
        torch.cuda.empty_cache()

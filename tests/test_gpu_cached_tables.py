"""MI355_OPT_CACHE_KERNELS over calls whose kernels read different table
layouts (gridding on bands, degridding, gridding on strips): each keeps its
tables while the stack's pointer and shape stay.  Shown by clearing the stack
in place, which a call that rebuilds its tables sees and one that keeps them
does not."""
import numpy as np
import pytest

from mi355_gridding import _lib, synth

pytestmark = pytest.mark.gpu


class _Calls:
    def __init__(self, torch, ops, ctx, c, dtype):
        self.torch, self.ops, self.ctx, self.c = torch, ops, ctx, c
        self.ks = ops.KernelStack(c["support"], c["oversample"], c["conv_size_half"],
                                  c["conv_func"], dtype=dtype)
        self.d = {k: torch.from_numpy(np.ascontiguousarray(c[k])).cuda().to(dtype)
                  for k in ("uu", "vv", "ww", "vis", "weight")}
        G = c["grid_size"]
        rng = np.random.default_rng(2)
        self.g0 = torch.from_numpy(rng.normal(size=(G, G, 2))).cuda().to(dtype)

    def grid(self):
        c, d, torch = self.c, self.d, self.torch
        grid = torch.zeros_like(self.g0)
        norm = torch.zeros(1, dtype=torch.float64, device="cuda")
        sk = torch.zeros(1, dtype=torch.int64, device="cuda")
        self.ops.grid(self.ks, d["uu"], d["vv"], d["ww"], d["vis"], d["weight"],
                      c["cell_size_rad"], c["w_scale"], c["grid_size"], grid, norm, sk,
                      ctx=self.ctx)
        return torch.cat([grid.double().flatten(), norm])

    def degrid(self):
        c, d = self.c, self.d
        return self.ops.degrid(self.ks, d["uu"], d["vv"], d["ww"], d["weight"],
                               c["cell_size_rad"], c["w_scale"], c["grid_size"], self.g0,
                               ctx=self.ctx).double().flatten()

    def strips(self):
        self.ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 6)
        try:
            return self.grid()
        finally:
            self.ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 0)


def _context(torch, **opts):
    ctx = _lib.Context(torch.cuda.current_device())
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    for k, v in opts.items():
        ctx.set_option(getattr(_lib, k), v)
    return ctx


@pytest.mark.parametrize("double", [False, True])
def test_alternating_calls_keep_their_tables(gpu, double):
    torch, ops = gpu
    dtype = torch.float64 if double else torch.float32
    c = synth.make(0, num_points=6000, grid_size=512, num_w_planes=32, max_support=14, seed=41)
    other = synth.make(0, num_points=3000, grid_size=512, num_w_planes=24, max_support=9, seed=42)
    ctx = _context(torch, OPT_CACHE_KERNELS=1)
    try:
        a, b = _Calls(torch, ops, ctx, c, dtype), _Calls(torch, ops, ctx, other, dtype)
        calls = [a.grid, a.degrid] + ([] if double else [a.strips])
        first = [f() for f in calls]
        assert all(x.abs().max() > 0 for x in first)
        a.ks.conv.zero_()
        for _ in range(2):
            assert all(torch.equal(f(), x) for f, x in zip(calls, first))
        # another stack: every set goes, so that the next calls see the cleared one
        assert b.grid().abs().max() > 0
        assert all(f().abs().max() == 0 for f in calls)
        # as does setting the option
        a.ks.conv.fill_(1)
        assert all(f().abs().max() == 0 for f in calls)
        ctx.set_option(_lib.OPT_CACHE_KERNELS, 1)
        assert all(f().abs().max() > 0 for f in calls)
    finally:
        ctx.close()


def test_cached_sets_give_way_to_a_workspace_cap(gpu):
    """Tables of about 40 MiB in either layout under a cap of 56 MiB: the set
    not in use is given back, and alternating calls go on as without a cap."""
    torch, ops = gpu
    c = synth.make(0, num_points=2000, grid_size=512, num_w_planes=64, max_support=60, seed=43)
    free = _context(torch)
    ctx = _context(torch, OPT_CACHE_KERNELS=1, OPT_MAX_WORKSPACE=56 << 20,
                   OPT_VISITS_PER_ITEM=1024)
    try:
        want = _Calls(torch, ops, free, c, torch.float32)
        free.set_option(_lib.OPT_VISITS_PER_ITEM, 1024)
        a = _Calls(torch, ops, ctx, c, torch.float32)
        for _ in range(3):
            assert torch.equal(a.grid(), want.grid())
            assert torch.equal(a.degrid(), want.degrid())
    finally:
        ctx.close()
        free.close()

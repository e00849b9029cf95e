"""Timed cases of the gridder: what its users have it do, through the public
torch entry points (mi355_gridding.torch_ops), over the sizes they use.

A case is a plain dict; its "kind" names the entry point:

  grid      torch_ops.grid: one image's visibilities onto a cleared grid
  batched   torch_ops.grid_batched: many independent grids in one call
  degrid    torch_ops.degrid: predicted visibilities from a grid
  step      torch_ops.grid_autograd, forward and backward
  weights   torch_ops.grid_weights_write + grid_weights_read
  image     torch_ops.grid_to_image

Workloads follow the repository's synthetic data sets (csrc/synth.cpp):
radii from an exponential or a log-normal law, ww ~ N(0, (0.3 r)^2),
independent samples or baselines followed over one-minute steps, a
Gaussian-tapered chirp per w-plane with supports growing to `smax`.  Inputs
are drawn on the GPU from the seed.  The repository's root is the working
folder; the package lies in gpu-gridding_amd/ below it.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpu-gridding_amd"))

from mi355_gridding import _lib, synth, torch_ops as ops  # noqa: E402

UMAX = 1.0e4          # longest baseline, wavelengths (csrc/synth.cpp)


def _case(kind, **kw):
    c = dict(kind=kind, n=0, times=1, G=0, P=0, smax=0, ov=4, dist=0, double=False,
             compensated=False, jobs=1)
    c.update(kw)
    return c


def listed():
    return [
        # A few baselines onto a small odd-sized grid: what one interactive or
        # unit-sized call costs, launches and host work above all.
        _case("grid", name="grid_2k_301", n=2003, G=301, P=16, smax=8),
        # The 200k-visibility data set: a small field, one call.
        _case("grid", name="grid_200k_2048", n=200_000, G=2048, P=64, smax=16),
        # The synthetic challenge set (2,152,800 visibilities, 714 planes).
        _case("grid", name="grid_2m_8192", n=21_528 * 100, times=100, G=8192, P=714, smax=36),
        # The SKA-LOW set (31,395,840 visibilities, 601 planes, support 72),
        # the largest single-grid call.
        _case("grid", name="grid_31m_16384", n=130_816 * 240, times=240, G=16384, P=601, smax=72,
              dist=1),
        # Compensated FP32 accumulation, for deep integrations.
        _case("grid", name="grid_comp_1m_4096", n=1_000_000, G=4096, P=128, smax=32,
              compensated=True),
        # Double precision: one block of the synthetic set, as the driver
        # hands blocks over.
        _case("grid", name="grid_f64_215k_8192", n=21_528 * 10, times=10, G=8192, P=714, smax=36,
              double=True),
        # Snapshots / channels sharing one kernel stack, of uneven sizes.
        _case("batched", name="batched_24x4096", n=50_000, jobs=24, G=4096, P=339, smax=44),
        # Prediction from a model grid.
        _case("degrid", name="degrid_1m_4096", n=1_000_000, G=4096, P=128, smax=32),
        # The same in double precision, ragged, on an odd grid.
        _case("degrid", name="degrid_f64_100k_2047", n=100_003, G=2047, P=64, smax=16, double=True),
        # One optimisation step through the gridder: grid, norm and the
        # gradients of amplitudes and weights.
        _case("step", name="step_1m_4096", n=1_000_000, G=4096, P=128, smax=32),
        # Uniform weighting of the SKA-LOW set: density, then the weights.
        _case("weights", name="weights_31m_16384", n=130_816 * 240, times=240, G=16384, smax=72,
              dist=1),
        # The dirty image of an 8192^2 grid.
        _case("image", name="image_8192", G=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _table_bytes(c):
    """Size of the kernel tables expanded per offset pair, from above."""
    w = 2 * c["smax"] + 1
    return c["P"] * (w + 14) * w * ((c["ov"] + 1) // 2 + 1) ** 2 * (16 if c["double"] else 8)


def draw(rng):
    kind = rng.choice(["grid"] * 8 + ["batched", "degrid", "degrid", "degrid", "step", "weights",
                                      "weights", "image"])
    if kind == "image":
        return _case("image", G=2 * _log_int(rng, 64, 8192), double=rng.random() < 0.25)
    if kind == "weights":
        times = rng.choice([1, 1, 10, 100])
        return _case("weights", n=max(1, _log_int(rng, 1000, 31_000_000) // times) * times,
                     times=times, G=_log_int(rng, 256, 16384), smax=8, dist=rng.choice([0, 1]),
                     double=rng.random() < 0.25)
    opt = rng.random()
    double = kind in ("grid", "degrid") and opt < 0.25
    comp = kind == "grid" and opt > 0.85
    c = _case(kind, G=_log_int(rng, 256, 16384 if kind == "grid" else 4096),
              P=_log_int(rng, 8, 714), ov=rng.choice([4, 4, 4, 4, 3, 2, 8]),
              dist=rng.choice([0, 1]), double=double, compensated=comp)
    c["smax"] = rng.randint(6, max(6, min(72, c["G"] // 8)))
    while _table_bytes(c) > 1.2e9:
        c["P"] = max(1, c["P"] // 2)
    # footprint taps of the whole call: below those of the largest listed
    # case, and of double precision, compensated and adjoint calls an eighth
    taps = (1.2 * c["smax"] + 1) ** 2
    most = (1.0e11 if kind in ("grid", "batched") and not (double or comp) else 1.2e10) / taps
    if kind == "batched":
        c["jobs"] = rng.randint(2, 24)
        c["n"] = _log_int(rng, 500, max(1000, min(50_000, most / (8 * c["jobs"]))))
        return c
    c["times"] = rng.choice([1, 1, 10, 100, 240])
    n = _log_int(rng, 1000, max(2000, min(31_000_000 if kind == "grid" else 2_000_000, most)))
    c["n"] = max(1, n // c["times"]) * c["times"]
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _job_counts(c):
    """Visibilities per job: from n to 40 n, evenly over the logarithm, the
    jobs in an order that mixes large and small ones."""
    k = c["jobs"]
    sizes = [int(c["n"] * 40.0 ** (j / max(1, k - 1))) | 1 for j in range(k)]
    return [sizes[(7 * j) % k if k % 7 else (5 * j + j // 5) % k] for j in range(k)]


def _coords(gen, n, times, dist, real):
    """uu, vv, ww of n samples (csrc/synth.cpp's laws)."""
    dev = "cuda"
    m = n // times
    u = torch.rand(m, generator=gen, device=dev, dtype=torch.float64)
    if dist == 0:
        r = -torch.log(1.0 - u) * (0.15 * UMAX)
    else:
        r = (0.05 * UMAX) * torch.exp(1.2 * torch.randn(m, generator=gen, device=dev,
                                                        dtype=torch.float64))
        r = r.clamp(max=UMAX)
    theta = 2 * math.pi * torch.rand(m, generator=gen, device=dev, dtype=torch.float64)
    w0 = 0.3 * r * torch.randn(m, generator=gen, device=dev, dtype=torch.float64)
    step = 2 * math.pi * 60.0 / 86400.0
    ha = (torch.arange(times, device=dev, dtype=torch.float64) - 0.5 * (times - 1)) * step
    ha = ha[:, None]                                     # time-major, as a block holds them
    uu = (r * torch.cos(theta + ha)).to(real).reshape(-1)
    vv = (r * torch.sin(theta + ha)).to(real).reshape(-1)
    ww = (w0 + 0.05 * r * torch.sin(ha)).to(real).reshape(-1)
    return uu, vv, ww


def _w_scale(ww, P):
    """(P - 1)^2 over the 99.9th percentile of |ww| (of a million samples)."""
    a = torch.sort(ww[:: max(1, ww.numel() // 1_000_000)].abs())[0]
    ref = float(a[int(0.999 * (a.numel() - 1))].item())
    return float(np.float32((P - 1) ** 2 / (ref if ref > 0 else 1.0)))


def _cell(c):
    return float(np.float32((c["G"] / 2 - c["smax"] - 2) / (UMAX * c["G"])))


def _real(c):
    return torch.float64 if c["double"] else torch.float32


def _samples(gen, n, times, c):
    real = _real(c)
    uu, vv, ww = _coords(gen, n, times, c["dist"], real)
    vis = torch.randn((n, 2), generator=gen, device="cuda", dtype=real) * math.sqrt(0.5)
    weight = 0.5 + torch.rand(n, generator=gen, device="cuda", dtype=real)
    return dict(uu=uu, vv=vv, ww=ww, vis=vis, weight=weight)


def _stack(c):
    support, conv, csh = synth.kernels(c["P"], c["smax"], c["ov"])
    return ops.KernelStack(support, c["ov"], csh, conv, dtype=_real(c))


_comp_ctx = []


def _context(c):
    """The context a call runs on: the package's own, or one kept for
    compensated accumulation."""
    if not c["compensated"]:
        return None
    if not _comp_ctx:
        _comp_ctx.append(_lib.Context(torch.cuda.current_device()))
        _comp_ctx[0].set_option(_lib.OPT_COMPENSATED, 1)
    _comp_ctx[0].set_stream(torch.cuda.current_stream().cuda_stream)
    return _comp_ctx[0]


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    real, G = _real(c), c["G"]
    s = dict(case=c, kind=c["kind"], G=G)
    z = dict(device="cuda")
    if c["kind"] == "image":
        s["grid"] = torch.randn((G, G, 2), generator=gen, dtype=real, **z)
        s["image"] = torch.empty((G, G), dtype=real, **z)
        s["norm"] = 0.5 * G
        return s
    s["skipped"] = torch.zeros(1, dtype=torch.int64, **z)
    s["cell"] = _cell(c)
    if c["kind"] == "weights":
        uu, vv, _ = _coords(gen, c["n"], c["times"], c["dist"], real)
        s.update(uu=uu, vv=vv, weight=0.5 + torch.rand(c["n"], generator=gen, dtype=real, **z),
                 weight_out=torch.zeros(c["n"], dtype=real, **z),
                 grid=torch.zeros((G, G), dtype=real, **z),
                 skipped2=torch.zeros(1, dtype=torch.int64, **z))
        return s
    s["ks"] = _stack(c)
    if c["kind"] == "batched":
        parts = [_samples(gen, k, 1, c) for k in _job_counts(c)]
        for k in ("uu", "vv", "ww", "vis", "weight"):
            s[k] = torch.cat([p[k] for p in parts])
        s["grids"] = torch.zeros((c["jobs"], G, G, 2), dtype=real, **z)
        s["norm"] = torch.zeros(c["jobs"], dtype=torch.float64, **z)
        s["skipped"] = torch.zeros(c["jobs"], dtype=torch.int64, **z)
        s["jobs"], off = [], 0
        for j, p in enumerate(parts):
            n = p["uu"].numel()
            s["jobs"].append(dict(vis_offset=off, num_points=n, cell_size_rad=s["cell"],
                                  w_scale=_w_scale(p["ww"], c["P"]), grid_size=G,
                                  grid=s["grids"][j], norm=s["norm"][j:j + 1],
                                  num_skipped=s["skipped"][j:j + 1]))
            off += n
        return s
    s.update(_samples(gen, c["n"], c["times"], c))
    s["w_scale"] = _w_scale(s["ww"], c["P"])
    if c["kind"] == "grid":
        s["grid"] = torch.zeros((G, G, 2), dtype=real, **z)
        s["norm"] = torch.zeros(1, dtype=torch.float64, **z)
        s["ctx"] = _context(c)
    else:
        # the model grid that is degridded / the gradient with respect to the grid
        s["model"] = torch.randn((G, G, 2), generator=gen, dtype=real, **z)
        if c["kind"] == "degrid":
            s["out"] = torch.empty((c["n"], 2), dtype=real, **z)
        else:
            s["vis"].requires_grad_(True)
            s["weight"].requires_grad_(True)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "grid":
        s["grid"].zero_()
        s["norm"].zero_()
        ops.grid(s["ks"], s["uu"], s["vv"], s["ww"], s["vis"], s["weight"], s["cell"],
                 s["w_scale"], s["G"], s["grid"], s["norm"], s["skipped"], ctx=s["ctx"])
        return dict(grid=s["grid"], norm=s["norm"], skipped=s["skipped"])
    if kind == "batched":
        s["grids"].zero_()
        s["norm"].zero_()
        ops.grid_batched(s["ks"], s["jobs"], s["uu"], s["vv"], s["ww"], s["vis"], s["weight"])
        return dict(grids=s["grids"], norm=s["norm"], skipped=s["skipped"])
    if kind == "degrid":
        return ops.degrid(s["ks"], s["uu"], s["vv"], s["ww"], s["weight"], s["cell"],
                          s["w_scale"], s["G"], s["model"], out=s["out"])
    if kind == "step":
        grid, norm = ops.grid_autograd(s["vis"], s["weight"], s["ks"], s["uu"], s["vv"], s["ww"],
                                       s["cell"], s["w_scale"], s["G"])
        gv, gw = torch.autograd.grad(grid, (s["vis"], s["weight"]), grad_outputs=s["model"])
        return dict(grid=grid.detach(), norm=norm.detach(), grad_vis=gv, grad_weight=gw)
    if kind == "weights":
        s["grid"].zero_()
        ops.grid_weights_write(s["uu"], s["vv"], s["weight"], s["cell"], s["G"], s["grid"],
                               s["skipped"])
        ops.grid_weights_read(s["uu"], s["vv"], s["weight"], s["weight_out"], s["cell"], s["G"],
                              s["grid"], s["skipped2"])
        return dict(grid=s["grid"], weight=s["weight_out"], skipped=s["skipped"],
                    skipped2=s["skipped2"])
    ops.grid_to_image(s["grid"], s["G"], s["image"], norm=s["norm"])
    return s["image"]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _supports(c):
    k = np.arange(c["P"])
    f = np.sqrt(k / (c["P"] - 1)) if c["P"] > 1 else np.ones(1)
    return np.clip(np.ceil(4.0 + (c["smax"] - 4) * f - 1e-12), 1, c["smax"]).astype(np.int64)


def _mean_taps(c):
    """Mean footprint taps of a visibility, from 200,000 samples of the law."""
    rng = np.random.default_rng(1)
    m = 200_000
    r = -np.log(1.0 - rng.random(m)) * 0.15 * UMAX if c["dist"] == 0 else \
        np.minimum(0.05 * UMAX * np.exp(1.2 * rng.normal(size=m)), UMAX)
    th = 2 * np.pi * rng.random(m)
    w = np.abs(0.3 * r * rng.normal(size=m))
    scale = (c["P"] - 1) ** 2 / max(np.quantile(w, 0.999), 1e-30)
    s = _supports(c)[np.minimum(np.round(np.sqrt(w * scale)), c["P"] - 1).astype(np.int64)]
    reach = (c["G"] / 2 - c["smax"] - 2) / UMAX
    inside = (np.abs(r * np.cos(th)) * reach + s < c["G"] / 2 - 1) & \
        (np.abs(r * np.sin(th)) * reach + s < c["G"] / 2 - 1)
    return float(np.mean(np.where(inside, (2 * s + 1) ** 2, 0)))


def work(case):
    c = case
    f = 8 if c["double"] else 4
    cells = float(c["G"]) ** 2
    if c["kind"] == "image":
        # a real image of a complex grid: half a complex transform's operations
        return dict(bytes=3 * f * cells, flops=2.5 * cells * math.log2(cells))
    if c["kind"] == "weights":
        # write: three arrays in, the grid out; read: three in and the grid, one out
        return dict(bytes=7 * f * c["n"] + 2 * f * cells, flops=2.0 * c["n"])
    # the part of the kernel stack that the supports reach, in samples per plane
    stack = 2 * f * float(np.sum((c["ov"] * _supports(c) + (c["ov"] + 1) // 2 + 1) ** 2))
    n = sum(_job_counts(c)) if c["kind"] == "batched" else c["n"]
    flops = 8.0 * n * _mean_taps(c)
    grid = 2 * f * cells * c["jobs"]
    if c["kind"] == "degrid":
        return dict(bytes=6 * f * n + stack + grid, flops=flops)
    if c["kind"] == "step":
        # coordinates, amplitudes and weights in, their gradients out, the
        # gradient of the grid in and the grid out
        return dict(bytes=9 * f * n + stack + 2 * grid, flops=2 * flops)
    return dict(bytes=6 * f * n + stack + grid, flops=flops)


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _round(x):
    """Half away from zero, exactly."""
    t = torch.trunc(x)
    return t + torch.sign(x) * ((x - t).abs() >= 0.5).to(x.dtype)


def _cells(c, uu, vv, cell):
    """Cell, and offset before rounding, per axis: in the inputs' precision."""
    one = np.float64 if c["double"] else np.float32
    gs = float(one(c["G"]) * one(cell))
    pu, pv = -uu * gs, vv * gs
    ru, rv = _round(pu), _round(pv)
    half = c["G"] // 2
    return ru.long() + half, rv.long() + half, ru - pu, rv - pv


def _selection(c, d, cell, w_scale, support):
    gu, gv, fu, fv = _cells(c, d["uu"], d["vv"], cell)
    ou, ov = _round(fu * c["ov"]).long(), _round(fv * c["ov"]).long()
    x = (d["ww"] * w_scale).abs()
    root = torch.sqrt(x.double()).to(x.dtype)         # correctly rounded
    plane = _round(root).long().clamp(max=c["P"] - 1)
    s = support[plane]
    G = c["G"]
    skip = (gu + s >= G) | (gu - s < 0) | (gv + s >= G) | (gv - s < 0)
    return gu, gv, ou, ov, plane, s, skip


def _footprints(c, d, ks, cell, w_scale):
    """Chunks of visibilities of one support: their indices, the cells
    [B, W, W] of their footprints and the taps there (complex128)."""
    support = torch.from_numpy(ks.support.astype(np.int64)).cuda()
    gu, gv, ou, ov, plane, s, skip = _selection(c, d, cell, w_scale, support)
    csh = ks.conv_size_half
    conv = torch.view_as_complex(ks.conv.view(-1, 2).double())
    keep = torch.nonzero(~skip).view(-1)
    keep = keep[torch.argsort(plane[keep])]
    at = s[keep]
    for sup in torch.unique(at).tolist():
        idx = keep[at == sup]
        k = torch.arange(-sup, sup + 1, device="cuda")
        step = max(1, (1 << 24) // (2 * sup + 1) ** 2)
        for b in range(0, idx.numel(), step):
            i = idx[b:b + step]
            iu = (ou[i][:, None] + c["ov"] * k).abs()
            iv = (ov[i][:, None] + c["ov"] * k).abs()
            taps = conv[(plane[i] * csh * csh)[:, None, None] + iv[:, :, None] * csh + iu[:, None]]
            conj = (d["ww"][i] > 0)[:, None, None]
            taps = torch.where(conj, taps.conj().resolve_conj(), taps)
            cells = (gv[i][:, None] + k)[:, :, None] * c["G"] + (gu[i][:, None] + k)[:, None, :]
            yield i, cells, taps
    yield torch.nonzero(skip).view(-1), None, None


def _exact_grid(c, d, ks, cell, w_scale):
    G = c["G"]
    grid = torch.zeros((G * G, 2), dtype=torch.float64, device="cuda")
    norm = torch.zeros((), dtype=torch.float64, device="cuda")
    amp = torch.view_as_complex(d["vis"].detach().double() * d["weight"].detach().double()[:, None])
    for i, cells, taps in _footprints(c, d, ks, cell, w_scale):
        if cells is None:
            return grid.view(G, G, 2), norm.view(1)
        grid.index_add_(0, cells.reshape(-1),
                        torch.view_as_real(taps * amp[i][:, None, None]).reshape(-1, 2))
        norm += (taps.real.sum(dim=(1, 2)) * d["weight"].detach()[i].double()).sum()


def _exact_degrid(c, d, ks, cell, w_scale, model):
    """sum over each footprint of conj(tap) * grid (no weight)."""
    g = torch.view_as_complex(model.double()).reshape(-1)
    out = torch.zeros(d["uu"].numel(), dtype=torch.complex128, device="cuda")
    for i, cells, taps in _footprints(c, d, ks, cell, w_scale):
        if cells is not None:
            out[i] = (taps.conj() * g[cells]).sum(dim=(1, 2))
    return torch.view_as_real(out)


def exact(case, seed):
    c = case
    if c["kind"] not in ("image", "weights"):
        n = sum(_job_counts(c)) if c["kind"] == "batched" else c["n"]
        if n * _mean_taps(c) > 1.0e10:
            return None
    s = prepare(c, seed)
    if c["kind"] == "image":
        g = torch.view_as_complex(s["grid"].double())
        g = torch.fft.ifftshift(g)
        img = torch.fft.fftshift(torch.fft.ifft2(g, norm="forward"))
        return img.real / s["norm"]
    if c["kind"] == "weights":
        G = c["G"]
        gu, gv, _, _ = _cells(c, s["uu"], s["vv"], s["cell"])
        ok = (gu >= 0) & (gu < G) & (gv >= 0) & (gv < G)
        at = (gv * G + gu)[ok]
        w = s["weight"].double()
        grid = torch.zeros(G * G, dtype=torch.float64, device="cuda").index_add_(0, at, w[ok])
        out = torch.zeros_like(w)
        out[ok] = w[ok] / grid[at]
        return dict(grid=grid.view(G, G), weight=out, skipped=None, skipped2=None)
    if c["kind"] == "batched":
        grids, norms = [], []
        for j in s["jobs"]:
            a, b = j["vis_offset"], j["vis_offset"] + j["num_points"]
            d = {k: s[k][a:b] for k in ("uu", "vv", "ww", "vis", "weight")}
            g, nm = _exact_grid(c, d, s["ks"], s["cell"], j["w_scale"])
            grids.append(g)
            norms.append(nm)
        return dict(grids=torch.stack(grids), norm=torch.cat(norms), skipped=None)
    if c["kind"] == "grid":
        g, nm = _exact_grid(c, s, s["ks"], s["cell"], s["w_scale"])
        return dict(grid=g, norm=nm, skipped=None)
    y = _exact_degrid(c, s, s["ks"], s["cell"], s["w_scale"], s["model"])
    if c["kind"] == "degrid":
        return y * s["weight"].double()[:, None]
    g, nm = _exact_grid(c, s, s["ks"], s["cell"], s["w_scale"])
    w, v = s["weight"].detach().double(), s["vis"].detach().double()
    return dict(grid=g, norm=nm, grad_vis=y * w[:, None], grad_weight=(v * y).sum(dim=1))

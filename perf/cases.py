"""Performance cases: what a user of this library has it do, through its public
Python entry points, over the sizes that its configurations, tests and
benchmark use.

A case is a dict of plain values; ``kind`` names the path:

  chunk        DdtrPlan.execute_chunk: one time chunk of one beam, corner turn,
               binning levels and every DM range (8- and 16-bit samples)
  batch        DdtrBatch.execute: many small beams, replayed from a hipGraph
  pipeline     aa_py_pipeline over host samples, planes back on the host
  outliers     zero_dm_outliers on a chunk that has just arrived
  condition    zero_dm and input normalisation of a chunk, output
               normalisation of a DM-time plane
  spd          spd_first_pass on one DM-time plane
  frac         frac_dedisperse, forward and backward (gradients of windows and DMs)
  refine       RefinePlan.run: coarse scan and gradient steps of many windows

DM ranges are written ``low-high/step/bin`` with commas between them.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "astro-accelerate_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import py_astro_accelerate as aa  # noqa: E402
import frac_ddtr  # noqa: E402
import multibeam  # noqa: E402

DEV = "cuda:0"
TSAMP = 64e-6
FREE_MEMORY = 64 << 30
PLAN_8 = ("0-150/0.1/1,150-300/0.2/1,300-500/0.25/1,500-900/0.4/2,900-1200/0.6/4,1200-1500/0.8/4,"
          "1500-2000/1.0/4,2000-3000/2.0/8")


def listed():
    return [
        # One small beam (a station or a quick look): a few launches of little work, latency counts.
        dict(name="chunk_small", kind="chunk", bits=8, container=8, nchans=128, nsamp=16384, fch1=1760.0,
             band=810.0, ranges="0-50/0.5/1,50-100/1/2"),
        # The plain single-range plan: 512 channels, 1000 trials, no binning.
        dict(name="chunk_single_range", kind="chunk", bits=8, container=8, nchans=512, nsamp=131072, fch1=1550.0,
             band=300.0, ranges="0-500/0.5/1"),
        # Ragged sizes: a channel count that is no multiple of 16, an odd length, samples in the
        # u16 container that the reference's reader makes.
        dict(name="chunk_ragged", kind="chunk", bits=8, container=16, nchans=1003, nsamp=200003, fch1=1500.0,
             band=320.0, ranges="0-100/0.5/1,100-300/1/2,300-700/2/4"),
        # The 8-range survey plan at full size: the largest ordinary chunk.
        dict(name="chunk_8range", kind="chunk", bits=8, container=8, nchans=4096, nsamp=1048576, fch1=1760.0,
             band=810.0, ranges=PLAN_8),
        # 16-bit filterbank (also what 32-bit files are scaled to).
        dict(name="chunk_16bit", kind="chunk", bits=16, container=16, nchans=1024, nsamp=131072, fch1=1500.0,
             band=300.0, ranges="0-100/0.5/1,100-300/1/2"),
        # Many small beams of a multi-beam receiver, each with its own plan, in one graph.
        dict(name="batch_small_beams", kind="batch", beams=96, plan_seed=20261202),
        # A whole observation through the drop-in FFI: host samples in, host planes out.
        dict(name="pipeline_host", kind="pipeline", nchans=512, nsamp=65536, fch1=1550.0, band=300.0,
             ranges="0-250/0.5/1,250-500/1/2"),
        # Interference mitigation of an arriving chunk.
        dict(name="zero_dm_outliers", kind="outliers", bits=8, nchans=4096, nsamp=262144),
        # Zero-DM and the two normalisations, as the pipeline's options apply them.
        dict(name="condition", kind="condition", nchans=4096, nsamp=262144, ndms=1536, plane_nsamp=222656),
        # First single-pulse pass over the first range's plane of the 8-range plan.
        dict(name="spd_first_pass", kind="spd", ndms=1536, nsamp=890624, width=32),
        # Differentiable dedispersion of candidate windows, a training step's forward and backward.
        dict(name="frac_windows", kind="frac", batch=32, nchans=4096, nsamp=1024, trials=64, span=2.0),
        # DM refinement of a batch of uneven candidate windows.
        dict(name="refine_windows", kind="refine", windows=256, steps=20, scan=9, plan_seed=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chunk", "chunk", "chunk", "batch", "outliers", "condition", "spd", "frac", "refine",
                       "pipeline"])
    if kind == "chunk":
        bits = rng.choice([8, 8, 8, 16])
        nchans = _log(rng, 64, 4096 if bits == 8 else 1500)
        if rng.random() < 0.5:
            nchans = max(64, nchans // 16 * 16)
        nsamp = _log(rng, 20000, 400000 if bits == 8 else 150000)
        # a DM ceiling whose sweep leaves at least half of the samples
        fch1 = rng.choice([1400.0, 1550.0, 1760.0])
        band = rng.choice([300.0, 400.0]) if fch1 < 1700 else rng.choice([400.0, 810.0])
        per_dm = 4148.741601 * (1.0 / (fch1 - band) ** 2 - 1.0 / fch1 ** 2) / TSAMP
        top = min(1000.0, 0.25 * nsamp / per_dm)
        nr = rng.randint(1, 3)
        edges = {1: [0, 1], 2: [0, 0.4, 1], 3: [0, 0.2, 0.5, 1]}[nr]
        step = rng.choice([0.1, 0.2, 0.25, 0.5])
        while top / step > 1600:
            step *= 2
        parts = ["%g-%g/%g/%d" % (round(edges[i] * top, 2), round(edges[i + 1] * top, 2), step * 2 ** i, 2 ** i)
                 for i in range(nr)]
        return dict(kind="chunk", bits=bits, container=16 if bits == 16 else rng.choice([8, 8, 16]), nchans=nchans,
                    nsamp=nsamp, fch1=fch1, band=band, ranges=",".join(parts))
    if kind == "batch":
        return dict(kind="batch", beams=_log(rng, 8, 128), plan_seed=rng.randint(1, 10 ** 6))
    if kind == "pipeline":
        return dict(kind="pipeline", nchans=16 * rng.randint(8, 40), nsamp=_log(rng, 40000, 80000), fch1=1550.0,
                    band=300.0, ranges=rng.choice(["0-120/0.5/1", "0-100/0.25/1,100-300/1/2"]))
    if kind == "outliers":
        return dict(kind="outliers", bits=rng.choice([8, 8, 16]), nchans=_log(rng, 100, 8192),
                    nsamp=_log(rng, 1000, 120000))
    if kind == "condition":
        return dict(kind="condition", nchans=rng.choice([16, 1]) * _log(rng, 24, 256), nsamp=_log(rng, 4000, 262144),
                    ndms=64 * rng.randint(1, 24), plane_nsamp=_log(rng, 2000, 222656))
    if kind == "spd":
        return dict(kind="spd", ndms=64 * rng.randint(1, 24), nsamp=_log(rng, 2000, 400000),
                    width=rng.choice([32, 32, 32, 16, 8, 5]))
    if kind == "frac":
        return dict(kind="frac", batch=rng.randint(1, 32), nchans=_log(rng, 64, 4096), nsamp=4 * _log(rng, 32, 512),
                    trials=rng.randint(1, 64), span=2.0)
    return dict(kind="refine", windows=_log(rng, 16, 256), steps=rng.randint(5, 20), scan=rng.choice([0, 5, 9]),
                plan_seed=rng.randint(1, 10 ** 6))


# ------------------------------------------------------------------ geometry
def _ranges(case):
    out = []
    for part in case["ranges"].split(","):
        span, step, ib = part.split("/")
        low, high = span.split("-")
        out.append((float(low), float(high), float(step), int(ib), int(ib)))
    return out


def _metadata(case):
    return aa.make_metadata(case["nchans"], case["nsamp"], case["fch1"], -case["band"] / case["nchans"], TSAMP,
                            nbits=case.get("bits", 8))


def _dmshifts(case):
    """Delay in seconds per unit DM, float32, as the dedispersion plan defines it."""
    f = np.float32(case["fch1"]) + np.float32(-case["band"] / case["nchans"]) * np.arange(case["nchans"],
                                                                                        dtype=np.float32)
    f = f.astype(np.float64)
    return (np.float64(np.float32(4148.741601)) * (1.0 / f ** 2 - 1.0 / f[0] ** 2)).astype(np.float32)


def _geometry(case):
    """Per range (dm_low, dm_step, ndms, bin, output samples): whole blocks of 64
    trials, ranges that follow one another, one time chunk in granules of 224."""
    f32 = np.float32
    user = _ranges(case)
    ndms = [(int((f32(h) - f32(lo)) / f32(s)) + 63) // 64 * 64 for lo, h, s, _, _ in user]
    low = [f32(user[0][0])]
    for i, (_, _, s, _, _) in enumerate(user):
        low.append(low[i] + f32(ndms[i]) * f32(s))
    last = _dmshifts(case)[-1]

    def extent(i):
        return int(math.ceil((low[i] + f32(user[i][2]) * f32(ndms[i])) * last / f32(TSAMP)))

    high = [int((f32(extent(i)) / f32(u[3]) + f32(224)) / f32(224)) * 224 * u[3] for i, u in enumerate(user) if u[3] > 1]
    maxshift = (max(high) if high else extent(len(user) - 1)) + 224
    ib = user[-1][3]
    local = (case["nsamp"] - maxshift) // ib // 224 * 224 * ib
    return [(float(low[i]), u[2], ndms[i], u[3], local // u[3] // 224 * 224) for i, u in enumerate(user)]


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _noise(shape, seed, mean, sigma, top, dtype):
    """Rounded Gaussian noise clipped to [0, top]."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat, g, n = out.view(-1), _generator(seed), 1 << 28
    for at in range(0, flat.numel(), n):
        part = flat[at:at + n]
        part.copy_(torch.randn(part.numel(), generator=g, device=DEV).mul_(sigma).add_(mean).round_().clamp_(0, top))
    return out


def _samples(case, seed):
    """[t][c] samples with a dispersed boxcar pulse; 16-bit ones as int16 bit patterns."""
    if case.get("bits", 8) == 8:
        x = _noise((case["nsamp"], case["nchans"]), seed, 128.0, 16.0, 223, torch.uint8)
        amplitude = 32
    else:
        x = _noise((case["nsamp"], case["nchans"]), seed, 12000.0, 1500.0, 32000, torch.int16)
        amplitude = 600
    dm = 0.5 * _ranges(case)[-1][1]
    delay = torch.from_numpy(np.floor(_dmshifts(case) * np.float32(dm / TSAMP)).astype(np.int64)).to(DEV)
    t0 = max(1, (case["nsamp"] - int(delay[-1])) // 3)
    for k in range(8):
        rows = (t0 + k + delay).clamp_(max=case["nsamp"] - 1)
        x[rows, torch.arange(case["nchans"], device=DEV)] += amplitude
    return x.to(torch.int16) if case.get("container", 8) == 16 and x.dtype == torch.uint8 else x


def _refine_sizes(case):
    rng = np.random.default_rng(case["plan_seed"])
    n = case["windows"]
    nchans = [int(v) for v in rng.choice([1024, 1536, 2048, 2560, 3072, 3584, 4096], n)]
    nsamp = [int(v) for v in rng.choice([256, 512, 1024, 2048, 4096, 777], n)]
    return nchans, nsamp


def _frac_delays(case):
    return (_dmshifts(dict(nchans=case["nchans"], fch1=1760.0, band=810.0)) / np.float32(TSAMP)).astype(np.float32)


def _frac_inputs(case, seed):
    g = _generator(seed)
    b, c, t = case["batch"], case["nchans"], case["nsamp"]
    x = torch.randn((b, c, t), generator=g, device=DEV)
    dm = ((torch.rand(b, generator=g, device=DEV) - 0.5) * 2.0)
    ds = torch.from_numpy(_frac_delays(case).astype(np.float64)).to(DEV)
    pos = torch.arange(t, device=DEV, dtype=torch.float64)
    for i in range(b):
        centre = t / 2.0 + ds * float(dm[i])
        x[i] += (0.5 * torch.exp(-0.5 * ((pos[None, :] - centre[:, None]) / 4.0) ** 2)).float()
    return x, dm


def _trials(case):
    return np.linspace(-case["span"], case["span"], case["trials"]).astype(np.float32)


# ------------------------------------------------------------------ the cases
def prepare(case, seed):
    kind = case["kind"]
    if kind == "chunk":
        s = aa.aa_py_ddtr_strategy(aa.make_plan(_ranges(case)), _metadata(case), FREE_MEMORY)
        tps = [s.t_processed(r, 0) for r in range(s.nranges)]
        outs = [torch.empty((s.ndms(r), tps[r]), dtype=torch.float32, device=DEV) for r in range(s.nranges)]
        return dict(kind=kind, plan=aa.DdtrPlan.from_strategy(s, sample_bits=case["bits"]), x=_samples(case, seed),
                    tps=tps, outs=outs)
    if kind == "batch":
        specs = multibeam.small_multibeam_specs(case["plan_seed"])[:case["beams"]]
        for i, sp in enumerate(specs):
            sp["seed"] = (int(seed) * 1000003 + i) % (1 << 31)
        beams = multibeam.build_beams(specs, DEV)
        return dict(kind=kind, beams=beams, batch=aa.DdtrBatch([b.plan for b in beams]),
                    inputs=[b.d_input for b in beams], tps=[b.tps for b in beams], outs=[b.outs for b in beams])
    if kind == "pipeline":
        s = aa.aa_py_ddtr_strategy(aa.make_plan(_ranges(case)), _metadata(case), FREE_MEMORY)
        comps, opts = aa.aa_py_pipeline_components(), aa.aa_py_pipeline_component_options()
        comps.dedispersion = True
        opts.copy_ddtr_data_to_host = True
        return dict(kind=kind, host=_samples(case, seed).cpu().numpy(), md=_metadata(case), comps=comps, opts=opts,
                    ranges=_ranges(case), strategy=s)
    if kind == "outliers":
        if case["bits"] == 8:
            raw = _noise((case["nsamp"], case["nchans"]), seed, 100.0, 12.0, 255, torch.uint8)
        else:
            raw = _noise((case["nsamp"], case["nchans"]), seed, 12000.0, 1500.0, 32000, torch.int16)
        hit = torch.randint(0, case["nchans"], (max(1, case["nchans"] // 64),), generator=_generator(seed + 1),
                            device=DEV)
        raw[:, hit] += 60 if case["bits"] == 8 else 9000   # channels with interference
        band = torch.full((case["nchans"],), (2.0 ** case["bits"] - 1) / 2, device=DEV)
        return dict(kind=kind, raw=raw, work=torch.empty_like(raw), band=band, bits=case["bits"])
    if kind == "condition":
        return dict(kind=kind, x=_noise((case["nsamp"], case["nchans"]), seed, 128.0, 16.0, 255, torch.uint8),
                    band=torch.full((case["nchans"],), 127.5, device=DEV),
                    plane=torch.randn((case["ndms"], case["plane_nsamp"]), generator=_generator(seed + 1),
                                      device=DEV).mul_(0.25).add_(128.0))
    if kind == "spd":
        plane = torch.randn((case["ndms"], case["nsamp"]), generator=_generator(seed), device=DEV).mul_(0.25).add_(128.0)
        plane[case["ndms"] // 2, case["nsamp"] // 3:case["nsamp"] // 3 + 12] += 1.5
        return dict(kind=kind, plane=plane, width=case["width"], work=aa.spd_workspace(DEV))
    if kind == "frac":
        x, dm = _frac_inputs(case, seed)
        plan = frac_ddtr.FracPlan(_frac_delays(case), _trials(case), case["nsamp"], case["batch"])
        return dict(kind=kind, plan=plan, x=x.requires_grad_(True), dm=dm.requires_grad_(True))
    if kind == "refine":
        nchans, nsamp = _refine_sizes(case)
        n = len(nchans)
        sizes = [c * t for c, t in zip(nchans, nsamp)]
        xo = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
        tables, do, off = [], {}, 0
        for c in sorted(set(nchans)):
            tables.append(_frac_delays(dict(nchans=c)))
            do[c], off = off, off + c
        g = _generator(seed)
        r = np.random.default_rng(seed).uniform(-1.0, 1.0, n)
        x = torch.randn(int(sum(sizes)), generator=g, device=DEV)
        for b in range(n):
            w = x[int(xo[b]):int(xo[b]) + sizes[b]].view(nchans[b], nsamp[b])
            t = torch.arange(nsamp[b], device=DEV)
            ds = torch.from_numpy(_frac_delays(dict(nchans=nchans[b]))).to(DEV)
            w += 0.5 * torch.exp(-0.5 * ((t[None, :] - (nsamp[b] / 2.0 + ds * float(r[b]))[:, None]) / 4.0) ** 2)
        plan = frac_ddtr.RefinePlan(nchans, nsamp, xo, [do[c] for c in nchans])
        f64 = dict(dtype=torch.float64, device=DEV)
        return dict(kind=kind, plan=plan, x=x, ds=torch.from_numpy(np.concatenate(tables)).to(DEV),
                    u=torch.zeros(n, device=DEV), step=torch.zeros(n, device=DEV), prev=torch.zeros(n, **f64),
                    loss=torch.zeros(n, **f64), grad=torch.zeros(n, **f64), steps=case["steps"],
                    scan=(case["scan"], -1.0, 2.0 / (case["scan"] - 1)) if case["scan"] else None)
    raise ValueError(kind)


def run(state):
    kind = state["kind"]
    if kind == "chunk":
        state["plan"].execute_chunk(state["x"], state["tps"], state["outs"])
        return state["outs"]
    if kind == "batch":
        state["batch"].execute(state["inputs"], state["tps"], state["outs"])
        # the planes of one beam in twelve, each whole: at most 64 outputs are compared
        return [o for b in state["outs"][::12] for o in b]
    if kind == "pipeline":
        with aa.aa_py_pipeline(state["comps"], state["opts"], state["md"], state["host"], 0) as pipe:
            pipe.bind_ddtr_plan(aa.make_plan(state["ranges"]))
            while pipe.run():
                pass
            if pipe.status_code() < 0:
                raise RuntimeError("the pipeline failed")
            return pipe.output_planes(state["strategy"])
    if kind == "outliers":
        state["work"].copy_(state["raw"])   # the chunk arrives in the device buffer that is filtered in place
        aa.zero_dm_outliers(state["work"], state["band"], nbits=state["bits"])
        return state["work"]
    if kind == "condition":
        aa.zero_dm(state["x"], state["band"])
        aa.input_ddtr_normalization(state["x"])
        aa.output_ddtr_normalization(state["plane"])
        return [state["x"], state["plane"]]
    if kind == "spd":
        return aa.spd_first_pass(state["plane"], state["width"], work=state["work"])
    if kind == "frac":
        y = frac_ddtr.frac_dedisperse(state["x"], state["dm"], state["plan"])
        gx, gdm = torch.autograd.grad(y.square().sum(), (state["x"], state["dm"]))
        return [y, gx, gdm]
    if kind == "refine":
        state["u"].zero_()
        state["step"].fill_(0.1)
        state["prev"].zero_()
        state["plan"].run(state["x"], state["ds"], state["u"], state["step"], state["prev"], state["loss"],
                          state["grad"], nsteps=state["steps"], scan=state["scan"])
        return [state["u"], state["step"], state["prev"], state["loss"], state["grad"]]
    raise ValueError(kind)


def work(case):
    """Inputs read once and outputs written once; additions and multiplications of the sums."""
    kind = case["kind"]
    if kind in ("chunk", "pipeline"):
        outs = sum(nd * tp for _, _, nd, _, tp in _geometry(case))
        return dict(bytes=case["nsamp"] * case["nchans"] * (case.get("container", 8) // 8) + 4.0 * outs,
                    flops=float(case["nchans"]) * outs)
    if kind == "batch":
        total = dict(bytes=0.0, flops=0.0)
        for sp in multibeam.small_multibeam_specs(case["plan_seed"])[:case["beams"]]:
            one = work(dict(kind="chunk", nchans=sp["nchans"], nsamp=sp["nsamp"], fch1=sp["fch1"],
                            band=multibeam.BAND_WIDTH_MHZ, ranges=",".join("%g-%g/%g/%d" % r[:4] for r in sp["ranges"])))
            total = {k: total[k] + one[k] for k in total}
        return total
    if kind == "outliers":
        n = float(case["nsamp"]) * case["nchans"]
        return dict(bytes=2 * n * (case["bits"] // 8), flops=0.0)
    if kind == "condition":
        n, p = float(case["nsamp"]) * case["nchans"], float(case["ndms"]) * case["plane_nsamp"]
        return dict(bytes=4 * n + 8 * p, flops=0.0)
    if kind == "spd":
        n = float(case["ndms"]) * case["nsamp"]
        return dict(bytes=10 * n, flops=4 * n * case["width"])
    if kind == "frac":
        b, c, t, k = case["batch"], case["nchans"], case["nsamp"], case["trials"]
        # forward, gradient of the windows, gradient of the DMs: two taps each, a multiply and an add per tap
        return dict(bytes=4.0 * b * t * (3 * c + 2 * k), flops=12.0 * b * c * t * k)
    if kind == "refine":
        nchans, nsamp = _refine_sizes(case)
        n = float(sum(c * t for c, t in zip(nchans, nsamp)))
        # the windows do not fit the caches: each gradient step needs a pass, the scan and the powers one
        return dict(bytes=4 * n * (case["steps"] + 2), flops=n * (4 * case["scan"] + 8 * (case["steps"] + 1)))
    raise ValueError(kind)


# ---------------------------------------------------------------- 64-bit results
def _exact_chunk(case, seed):
    geometry = _geometry(case)
    if sum(nd * tp for _, _, nd, _, tp in geometry) * float(case["nchans"]) > 4e11:
        return None
    level = _samples(case, seed).t().contiguous()
    level = level.to(torch.int32)
    if case["bits"] == 16:
        level &= 0xFFFF
    shifts, outs, bin_now = _dmshifts(case), [], 1
    for low, step, nd, ib, tp in geometry:
        while bin_now < ib:
            n = level.shape[1] // 2
            level = (level[:, 0:2 * n:2] + level[:, 1:2 * n:2]) // 2
            bin_now *= 2
        tsamp = np.float32(TSAMP) * np.float32(ib)
        start, inc = np.float32(low) / tsamp, np.float32(step) / tsamp
        dm = (np.arange(nd).astype(np.float64) * np.float64(inc) + np.float64(start)).astype(np.float32)
        total = torch.zeros((nd, tp), dtype=torch.int64, device=DEV)
        for c in range(case["nchans"]):
            delay = torch.from_numpy((shifts[c] * dm).astype(np.int64)).to(DEV)
            total += level[c].unfold(0, tp, 1)[delay]
        outs.append(total.double() / case["nchans"] / ib)
    return outs


def _exact_frac(case, seed):
    b, c, t, k = case["batch"], case["nchans"], case["nsamp"], case["trials"]
    x, dm = _frac_inputs(case, seed)
    u = torch.from_numpy(_trials(case).astype(np.float64)).to(DEV)[None, :] + dm.double()[:, None]
    ds = _frac_delays(case).astype(np.float64)
    pos = torch.arange(t, device=DEV)

    def taps(ch):
        tau = float(ds[ch]) * u
        i0 = torch.floor(tau)
        return i0.long()[:, :, None], (tau - i0)[:, :, None]

    def at(rows, idx):
        # rows [b][1 or k][t] at positions idx [b][k][t], zero outside the window
        inside = (idx >= 0) & (idx < t)
        return torch.where(inside, torch.gather(rows.expand(b, k, t), 2, idx.clamp(0, t - 1)), 0.0)

    y = torch.zeros((b, k, t), dtype=torch.float64, device=DEV)
    for ch in range(c):
        i0, f = taps(ch)
        row = x[:, ch, None, :].double()
        y += (1 - f) * at(row, pos + i0) + f * at(row, pos + i0 + 1)
    gy, gdm = 2 * y, torch.zeros(b, dtype=torch.float64, device=DEV)
    gx = torch.empty((b, c, t), dtype=torch.float64, device=DEV)
    for ch in range(c):
        i0, f = taps(ch)
        row = x[:, ch, None, :].double()
        gx[:, ch] = ((1 - f) * at(gy, pos - i0) + f * at(gy, pos - i0 - 1)).sum(1)
        gdm += float(ds[ch]) * (gy * (at(row, pos + i0 + 1) - at(row, pos + i0))).sum((1, 2))
    return [y, gx, gdm]


def _exact_spd(case, seed):
    x = prepare(case, seed)["plane"]
    nd, n, w_max = case["ndms"], case["nsamp"], case["width"]
    blocks = [(at, min(nd, at + max(1, (1 << 27) // n))) for at in range(0, nd, max(1, (1 << 27) // n))]
    centre = float(x.double().mean()) if x.numel() < 1 << 28 else 128.0
    sums = torch.zeros((w_max, 2), dtype=torch.float64, device=DEV)
    for a, e in blocks:
        part = x[a:e].double() - centre
        box = torch.zeros_like(part)
        for w in range(1, w_max + 1):
            box[:, :n - w + 1] += part[:, w - 1:]
            v = box[:, :n - w + 1]
            sums[w - 1, 0] += v.sum()
            sums[w - 1, 1] += v.square().sum()
    count = torch.tensor([float(nd) * (n - w + 1) for w in range(1, w_max + 1)], device=DEV, dtype=torch.float64)
    mean = sums[:, 0] / count
    sd = (sums[:, 1] / count - mean ** 2).clamp(min=0).sqrt()
    snr = torch.full((nd, n), -math.inf, dtype=torch.float64, device=DEV)
    for a, e in blocks:
        part = x[a:e].double() - centre
        box = torch.zeros_like(part)
        for w in range(1, w_max + 1):
            v = box[:, :n - w + 1]
            v += part[:, w - 1:]
            best = snr[a:e, :n - w + 1]
            torch.maximum(best, (v - mean[w - 1]) / sd[w - 1], out=best)
    widths = torch.arange(1, w_max + 1, device=DEV, dtype=torch.float64)
    return [torch.stack([mean + widths * centre, sd], 1), snr, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "chunk":
        return _exact_chunk(case, seed)
    if kind == "pipeline":
        out = _exact_chunk(dict(case, bits=8, container=8), seed)
        return None if out is None else [o.cpu().numpy() for o in out]
    if kind == "condition":
        plane = prepare(case, seed)["plane"].double()
        return [None, plane - (plane.mean(0, keepdim=True) - 127.5)]
    if kind == "spd":
        return _exact_spd(case, seed)
    if kind == "frac":
        return _exact_frac(case, seed)
    return None

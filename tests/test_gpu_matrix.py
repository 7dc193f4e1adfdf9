"""The matrix-core dedispersion kernel (the automatic choice of a DdtrPlan
range whose channel groups fit it, unless it is as small as these), bit for bit
against the CPU oracle at the edges of its tiles, groups and steps; in a batch;
and over the byte planes of 16-bit samples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name, nchans, fch1, foff, dm_low, dm_step, ndms, t_processed, inBin, fill
GEOMS = [
    ("one_sample_last_tile", 512, 1550.0, -0.5859, 0.0, 0.1, 64, 2 * 1888 + 1, 1, "noise"),
    ("dm_zero_tile", 512, 1550.0, -0.5859, 0.0, 0.5, 32, 4000, 1, "noise"),         # base delays start at 0
    ("ragged_channels", 333, 1500.0, -0.96, 12.3, 0.3, 48, 3001, 1, "noise"),       # last step part empty
    ("ragged_trials", 512, 1550.0, -0.5859, 40.0, 0.5, 37, 2500, 1, "noise"),       # last DM tile part empty
    ("one_trial", 1024, 1550.0, -0.29, 100.0, 0.5, 1, 1000, 1, "noise"),
    ("saturated", 4096, 1760.0, -0.19775, 0.0, 0.1, 16, 2100, 1, "full"),           # largest sums, groups of 256
    ("zeros", 1024, 1760.0, -0.391, 10.0, 0.2, 16, 2100, 1, "zero"),                # every byte at the signed end
    ("two_windows", 512, 1550.0, -0.5859, 300.0, 1.0, 48, 3333, 1, "noise"),        # 8-byte windows
    ("four_windows", 416, 1760.0, -0.96, 500.0, 1.6, 32, 3000, 2, "noise"),         # 16-byte windows, binned
    ("many_channels", 16384, 1500.0, -0.0244140625, 0.0, 0.2, 20, 2500, 1, "noise"),
]


@pytest.mark.parametrize("pitch_extra", [0, 13])
@pytest.mark.parametrize("geom", GEOMS, ids=[g[0] for g in GEOMS])
def test_matrix_range(aa, oracle, cuda, geom, pitch_extra):
    import torch
    name, nchans, fch1, foff, low, step, ndms, tp, ib, fill = geom
    print(f"matrix {name} pitch +{pitch_extra}", flush=True)
    tsamp = 64e-6
    ds = oracle.dmshifts(nchans, fch1, foff)
    tsr = np.float32(np.float32(tsamp) * np.float32(ib))
    ms, st = np.float32(np.float32(low) / tsr), np.float32(np.float32(step) / tsr)
    maxd = int(np.trunc(np.float32(ds[-1]) * np.float32(np.float64(ndms - 1) * st + ms))) + 1
    nsamp = (tp + maxd) * ib
    rng = np.random.default_rng(nchans + ndms)
    if fill == "noise":
        data = rng.integers(0, 256, size=(nsamp, nchans), dtype=np.uint8)
    else:
        data = np.full((nsamp, nchans), 255 if fill == "full" else 0, dtype=np.uint8)
        data[rng.integers(0, nsamp, 50), rng.integers(0, nchans, 50)] = 128
    rows = oracle.corner_turn(data, nsamp, nchans)
    for _ in range(ib.bit_length() - 1):
        rows = oracle.bin2(rows, rows.shape[1] // 2)
    want = oracle.dedisperse(rows[:, :tp + maxd].copy(), ds, ndms, tp, float(ms), float(st), ib)
    plan = aa.DdtrPlan(ds, [(low, step, ndms, ib)], tsamp, maxd * ib, tp * ib)
    d_in = torch.from_numpy(data).to(cuda)
    for kernel in (aa.KERNEL_AUTO, aa.KERNEL_LDS, aa.KERNEL_MATRIX):
        plan.set_kernel(kernel)
        out = torch.full((ndms, tp + pitch_extra), -1.0, dtype=torch.float32, device=cuda)
        plan.ingest(d_in, tp * ib)
        plan.run_range(0, tp, out)
        ran = plan.range_kernel(0)
        assert ran == aa.RANGE_MATRIX if kernel == aa.KERNEL_MATRIX else ran != aa.RANGE_MATRIX
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[:, :tp], want)
        assert np.all(got[:, tp:] == -1.0)   # nothing written past a row's samples


def test_matrix_choice_follows_the_kernel_setting(aa, oracle, cuda):
    """The automatic choice, a forced shape and a preferred one, in turn on one handle."""
    import torch
    nchans, tsamp, tp, ndms = 512, 64e-6, 3000, 48
    ds = oracle.dmshifts(nchans, 1550.0, -0.5859)
    maxd = int(ds[-1] * (0.5 * ndms / tsamp)) + 2
    data = oracle.gen_noise(5, tp + maxd, nchans)
    plan = aa.DdtrPlan(ds, [(0.0, 0.5, ndms, 1)], tsamp, maxd, tp)
    d_in = torch.from_numpy(data).to(cuda)
    want = oracle.dedisperse(oracle.corner_turn(data, tp + maxd, nchans), ds, ndms, tp, 0.0,
                             float(np.float32(0.5) / np.float32(tsamp)), 1)
    plan.ingest(d_in, tp)
    for kernel, variant in ((0, -1), (5, -1), (0, -1), (0, 4), (0, 1), (0, -1), (1, -1), (2, -1), (7, -1)):
        plan.set_kernel(kernel)
        plan.set_range_variant(0, variant)
        out = torch.full((ndms, tp), -1.0, dtype=torch.float32, device=cuda)
        plan.run_range(0, tp, out)
        np.testing.assert_array_equal(out.cpu().numpy(), want, err_msg=f"kernel {kernel} variant {variant}")


def test_matrix_launches_of_a_batch(aa, oracle, cuda):
    """Ranges of at least 512 tiles run matrix launches of their own in a batch,
    eager and replayed with other inputs, beside ranges that share launches."""
    import torch
    nchans, tsamp, tp, small = 256, 64e-6, 33000, 3000
    ds = oracle.dmshifts(nchans, 1550.0, -1.17)
    ranges = [(0.0, 0.25, 512, 1), (128.0, 0.5, 64, 2)]
    maxd = (int(ds[-1] * (160.0 / tsamp)) + 4) // 2 * 2
    plans = [aa.DdtrPlan(ds, ranges, tsamp, maxd, tp) for _ in range(2)]
    tps = [tp, small]
    ins = [torch.empty((tp + maxd, nchans), dtype=torch.uint8, device=cuda) for _ in plans]
    outs = [[torch.empty((r[2], t), dtype=torch.float32, device=cuda) for r, t in zip(ranges, tps)] for _ in plans]
    batch = aa.DdtrBatch(plans)
    for call, graph in enumerate((False, True, True, True)):   # eager, captured, replayed twice
        datas = [oracle.gen_noise(10 * call + b, tp + maxd, nchans) for b in range(2)]
        for b in range(2):
            ins[b].copy_(torch.from_numpy(datas[b]))
            for o in outs[b]:
                o.fill_(-1.0)
        torch.cuda.synchronize()
        batch.execute(ins, [tps] * 2, outs, use_graph=graph)
        torch.cuda.synchronize()
        assert [p.range_kernel(0) for p in plans] == [aa.RANGE_MATRIX] * 2
        assert all(0 <= p.range_kernel(1) < aa.LDS_SHAPES for p in plans)
        for b in range(2):
            rows = oracle.corner_turn(datas[b], tp + maxd, nchans)
            for r, (low, step, nd, ib) in enumerate(ranges):
                rows = rows if ib == 1 else oracle.bin2(rows, rows.shape[1] // 2)
                tsr = np.float32(np.float32(tsamp) * np.float32(ib))
                want = oracle.dedisperse(rows[:, :tps[r] + maxd // ib].copy(), ds, nd, tps[r],
                                         float(np.float32(low) / tsr), float(np.float32(step) / tsr), ib)
                np.testing.assert_array_equal(outs[b][r].cpu().numpy(), want, err_msg=f"call {call} beam {b} range {r}")


def _u16_fill(kind, nsamp, nchans, rng):
    x = rng.integers(0, 2001, size=(nsamp, nchans))
    if kind == "bytes":            # low and high byte at their ends
        x = rng.choice([0, 255, 256, 257, 65280], size=(nsamp, nchans), p=[0.3, 0.3, 0.2, 0.199, 0.001])
    elif kind == "straddle":       # sums on both sides of 2^24 in every tile
        x = rng.integers(2 ** 25 // nchans - 20000, 20000, size=(nsamp, nchans))
    elif kind == "mixed":          # the end of the plane rounds, the rest does not
        x[nsamp * 7 // 10:] += 60000
    elif kind == "over":
        x = rng.integers(50000, 65536, size=(nsamp, nchans))
    elif kind == "edge":           # sums of exactly 2^24, and a few above
        x = np.full((nsamp, nchans), 2 ** 24 // nchans)
        x[rng.integers(0, nsamp, 3), rng.integers(0, nchans, 3)] += 1
    return x.astype(np.uint16)


@pytest.mark.parametrize("kind", ["low", "bytes", "straddle", "mixed", "over", "edge"])
@pytest.mark.parametrize("nchans", [1024, 1003])
def test_u16_byte_planes(aa, oracle, cuda, kind, nchans):
    """16-bit plans: exact integer sums over the byte planes, and the float sums
    in channel order wherever one passes 2^24 and the adds round."""
    import torch
    print(f"matrix u16 {kind} {nchans} channels", flush=True)
    ranges = [(0, 20, 0.4, 1, 1), (20, 45, 0.8, 2, 2)]
    tsamp, nsamp = 64e-6, 16000
    s = oracle.strategy(ranges, nchans, nsamp, 1500.0, -300.0 / nchans, tsamp, nbits=16)
    assert s.ok and s.num_tchunks == 1
    x = _u16_fill(kind, nsamp, nchans, np.random.default_rng(nchans))
    want = oracle.run(s, x)
    plan = aa.DdtrPlan(s.dmshifts, [(s.dm[r][0], s.dm[r][2], s.ndms[r], s.dm[r][3]) for r in range(s.nranges)],
                       tsamp, s.maxshift, s.t_processed[0][0], sample_bits=16)
    tps = [s.t_processed[r][0] for r in range(s.nranges)]
    d_in = torch.from_numpy(x.view(np.int16)).to(cuda)
    for chunk in range(2):         # the second chunk finds the first one's planes and flags
        outs = [torch.full((s.ndms[r], tps[r] + 3), -1.0, dtype=torch.float32, device=cuda) for r in range(s.nranges)]
        plan.execute_chunk(d_in if chunk else torch.flip(d_in, (0,)).contiguous(), tps, outs)
    for r in range(s.nranges):
        assert plan.range_kernel(r) == aa.RANGE_MATRIX
        got = outs[r].cpu().numpy()
        np.testing.assert_array_equal(got[:, :tps[r]], want[r], err_msg=f"range {r}")
        assert np.all(got[:, tps[r]:] == -1.0)


def test_u16_lengths_on_two_streams(aa, oracle, cuda):
    """Two lengths of one 16-bit range on two streams at once: the shorter call's
    samples sum exactly, the longer one's round from the middle of a tile on."""
    import torch
    nchans, tsamp, nsamp, ndms, lengths = 1024, 64e-6, 16000, 64, (600, 4000)
    ds = oracle.dmshifts(nchans, 1500.0, -300.0 / nchans)
    maxd = int(ds[-1] * (0.4 * ndms / tsamp)) + 2
    assert 600 + maxd < 1500
    rng = np.random.default_rng(8)
    x = rng.integers(0, 2001, size=(nsamp, nchans))
    x[1500:4000 + maxd] = rng.integers(0, 40001, size=(2500 + maxd, nchans))   # sums about 2e7
    d_in = torch.from_numpy(x.astype(np.uint16).view(np.int16)).to(cuda)
    plan = aa.DdtrPlan(ds, [(0.0, 0.4, ndms, 1)], tsamp, maxd, nsamp - maxd, sample_bits=16)
    plan.ingest(d_in, nsamp - maxd)
    want = []
    for tp in lengths:
        out = torch.empty((ndms, tp), dtype=torch.float32, device=cuda)
        plan.run_range(0, tp, out)
        assert plan.range_kernel(0) == aa.RANGE_MATRIX
        want.append(out)
    direct = aa.DdtrPlan(ds, [(0.0, 0.4, ndms, 1)], tsamp, maxd, nsamp - maxd, sample_bits=16)
    direct.set_kernel(aa.KERNEL_DIRECT)      # in channel order, whatever the sums
    direct.ingest(d_in, nsamp - maxd)
    for tp, w in zip(lengths, want):
        out = torch.empty((ndms, tp), dtype=torch.float32, device=cuda)
        direct.run_range(0, tp, out)
        assert torch.equal(out, w)
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in lengths], [[], []]
    for _ in range(20):
        for i, (tp, s) in enumerate(zip(lengths, streams)):
            with torch.cuda.stream(s):
                out = torch.empty((ndms, tp), dtype=torch.float32, device=cuda)
                plan.run_range(0, tp, out, stream=s)
                got[i].append(out)
    torch.cuda.synchronize()
    for outs, w in zip(got, want):
        for out in outs:
            assert torch.equal(out, w)

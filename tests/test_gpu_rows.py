"""Small and coarse ranges summed straight from the rows (the automatic choice
of a DdtrPlan range that is small or whose trials are far apart), bit for bit
against the CPU oracle at the edges of its tiles, waves and channel blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name, nchans, fch1, foff, dm_low, dm_step, ndms, t_processed, inBin, fill
GEOMS = [
    ("one_channel", 1, 1500.0, -1.0, 0.0, 1.0, 5, 100, 1, "noise"),
    ("fewer_channels_than_waves", 3, 1500.0, -50.0, 0.0, 1.0, 5, 1008, 1, "noise"),
    ("ragged_waves", 31, 1500.0, -9.7, 3.0, 1.0, 7, 1007, 1, "noise"),
    ("two_delay_blocks", 259, 1500.0, -1.1, 1.0, 0.7, 9, 1009, 1, "noise"),
    ("largest_16_bit_sums", 1024, 1500.0, -0.3, 0.0, 0.1, 16, 2100, 1, "full"),
    ("zeros", 1024, 1500.0, -0.3, 0.0, 0.1, 16, 500, 1, "zero"),
    ("second_channel_block", 1025, 1500.0, -0.3, 0.0, 0.2, 16, 2016, 1, "full"),
    ("three_channel_blocks", 2333, 1500.0, -0.13, 2.0, 0.2, 3, 1500, 1, "noise"),
    ("coarse", 400, 1550.0, -0.75, 0.0, 40.0, 24, 6000, 1, "noise"),
    ("coarse_binned", 208, 1760.0, -3.9, 10.0, 15.0, 40, 5001, 2, "noise"),
    ("one_sample", 64, 1500.0, -4.7, 0.0, 0.5, 40, 1, 1, "noise"),
]


def _case(oracle, geom):
    _, nchans, fch1, foff, low, step, ndms, tp, ib, fill = geom
    tsamp = 64e-6
    ds = oracle.dmshifts(nchans, fch1, foff)
    tsr = np.float32(np.float32(tsamp) * np.float32(ib))
    ms, st = np.float32(np.float32(low) / tsr), np.float32(np.float32(step) / tsr)
    maxd = int(np.trunc(np.float32(ds[-1]) * np.float32(np.float64(ndms - 1) * st + ms))) + 1
    nsamp = (tp + maxd) * ib
    rng = np.random.default_rng(nchans + ndms)
    data = rng.integers(0, 256, size=(nsamp, nchans), dtype=np.uint8)
    if fill != "noise":
        data[:] = 255 if fill == "full" else 0
        data[rng.integers(0, nsamp, 50), rng.integers(0, nchans, 50)] = 128
    rows = oracle.corner_turn(data, nsamp, nchans)
    for _ in range(ib.bit_length() - 1):
        rows = oracle.bin2(rows, rows.shape[1] // 2)
    want = oracle.dedisperse(rows[:, :tp + maxd].copy(), ds, ndms, tp, float(ms), float(st), ib)
    return data, ds, tsamp, maxd, want


@pytest.mark.parametrize("pitch_extra", [0, 13])
@pytest.mark.parametrize("geom", GEOMS, ids=[g[0] for g in GEOMS])
def test_range(aa, oracle, cuda, geom, pitch_extra):
    import torch
    name, nchans, _, _, low, step, ndms, tp, ib, _ = geom
    print(f"rows {name} pitch +{pitch_extra}", flush=True)
    data, ds, tsamp, maxd, want = _case(oracle, geom)
    plan = aa.DdtrPlan(ds, [(low, step, ndms, ib)], tsamp, maxd * ib, tp * ib)
    out = torch.full((ndms, tp + pitch_extra), -1.0, dtype=torch.float32, device=cuda)
    plan.ingest(torch.from_numpy(data).to(cuda), tp * ib)
    plan.run_range(0, tp, out)
    assert plan.range_kernel(0) == aa.RANGE_ROWS
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:, :tp], want)
    assert np.all(got[:, tp:] == -1.0)   # nothing written past a row's samples


def test_autotune_and_batch(aa, oracle, cuda):
    """Autotuning a range of this kind, and a batch of them (whose ranges that
    fit no shape go the same way), leave its results as they are."""
    import torch
    geom = next(g for g in GEOMS if g[0] == "coarse")
    _, nchans, _, _, low, step, ndms, tp, ib, _ = geom
    data, ds, tsamp, maxd, want = _case(oracle, geom)
    plan = aa.DdtrPlan(ds, [(low, step, ndms, ib)], tsamp, maxd * ib, tp * ib)
    d_in = torch.from_numpy(data).to(cuda)
    out = torch.full((ndms, tp), -1.0, dtype=torch.float32, device=cuda)
    plan.ingest(d_in, tp * ib)
    plan.autotune_range(0, tp, out, 2)
    out.fill_(-1.0)
    plan.run_range(0, tp, out)
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    plans = [aa.DdtrPlan(ds, [(low, step, ndms, ib)], tsamp, maxd * ib, tp * ib) for _ in range(3)]
    batch = aa.DdtrBatch(plans)
    outs = [torch.empty((ndms, tp), dtype=torch.float32, device=cuda) for _ in plans]
    for graph in (False, True, True, True):
        for o in outs:
            o.fill_(-1.0)
        batch.execute([d_in] * 3, [[tp]] * 3, [[o] for o in outs], use_graph=graph)
        assert all(p.range_kernel(0) == aa.RANGE_ROWS for p in plans)
        torch.cuda.synchronize()
        for o in outs:
            np.testing.assert_array_equal(o.cpu().numpy(), want)

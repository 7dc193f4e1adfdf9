"""GPU: the wide corner turn at channel counts that are no multiple of 16 and
at any input address, and its binned levels inside a plan, bit for bit against
the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsamp,nchans", [(16384, 1), (16385, 15), (17000, 33), (2049, 1003), (16400, 127), (8193, 257),
                                          (66561, 100), (33001, 257), (8195, 1003)])   # the wide path
@pytest.mark.parametrize("sample_bytes,offset", [(1, 0), (1, 1), (1, 2), (1, 3), (2, 0), (2, 2)])
def test_turn(aa, oracle, cuda, nsamp, nchans, sample_bytes, offset):
    """offset: bytes from an aligned address.  The samples around the chunk
    are above 255 and must not set the flag."""
    import torch
    rng = np.random.default_rng(nsamp + nchans)
    dt = np.uint8 if sample_bytes == 1 else np.uint16
    x = rng.integers(0, 256, size=(nsamp, nchans), dtype=dt)
    lead = offset // sample_bytes
    flat = np.full(lead + nsamp * nchans + 64, 0xAB if sample_bytes == 1 else 0xABCD, dtype=dt)
    flat[lead:lead + nsamp * nchans] = x.reshape(-1)
    d = torch.from_numpy(flat if sample_bytes == 1 else flat.view(np.int16)).to(cuda)
    view = d[lead:lead + nsamp * nchans].view(nsamp, nchans)
    pitch = (nsamp + 255) // 256 * 256
    out = torch.full((nchans, pitch), 0xAB, dtype=torch.uint8, device=cuda)
    err = torch.zeros(1, dtype=torch.int32, device=cuda)
    aa.corner_turn_levels(view, sample_bytes, nsamp, nchans, [out], [pitch], err)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:, :nsamp], x.T.astype(np.uint8))
    assert np.all(got[:, nsamp:] == 0xAB)
    assert int(err.item()) == 0
    if sample_bytes == 2:
        for where in ((0, 0), (nsamp - 1, nchans - 1), (nsamp // 2, nchans // 2)):
            view[where] = 300
            err.zero_()
            aa.corner_turn_levels(view, sample_bytes, nsamp, nchans, [out], [pitch], err)
            assert int(err.item()) == 1
            view[where] = 7


@pytest.mark.parametrize("nchans,bits", [(99, 8), (99, 16), (333, 8), (7, 16)])
def test_plan_levels(aa, oracle, cuda, nchans, bits):
    """Ranges at the first three binned levels of a plan whose channel count
    is no multiple of 16."""
    import torch
    tsamp, ndms, tp0 = 64e-6, 16, 4 * 1400
    ds = oracle.dmshifts(nchans, 1500.0, -300.0 / nchans)
    ranges = [(0.0, 0.5, ndms, 1), (8.0, 1.0, ndms, 2), (24.0, 2.0, ndms, 4)]
    maxd = (int(ds[-1] * (56.0 / tsamp)) + 8) // 4 * 4
    nsamp = tp0 + maxd
    rng = np.random.default_rng(nchans)
    data = rng.integers(0, 256, size=(nsamp, nchans)).astype(np.uint8 if bits == 8 else np.uint16)
    plan = aa.DdtrPlan(ds, ranges, tsamp, maxd, tp0)
    d_in = torch.from_numpy(data if bits == 8 else data.view(np.int16)).to(cuda)
    plan.ingest(d_in, tp0)
    rows = oracle.corner_turn(data.astype(np.uint8), nsamp, nchans)
    for r, (low, step, nd, ib) in enumerate(ranges):
        if r:
            rows = oracle.bin2(rows, rows.shape[1] // 2)
        tp = tp0 // ib
        tsr = np.float32(np.float32(tsamp) * np.float32(ib))
        want = oracle.dedisperse(rows[:, :tp + maxd // ib].copy(), ds, nd, tp, float(np.float32(low) / tsr),
                                 float(np.float32(step) / tsr), ib)
        out = torch.full((nd, tp), -1.0, dtype=torch.float32, device=cuda)
        plan.run_range(r, tp, out)
        np.testing.assert_array_equal(out.cpu().numpy(), want)

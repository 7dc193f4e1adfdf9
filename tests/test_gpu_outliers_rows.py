"""Zero-DM with outlier rejection on 8-bit rows held in registers, bit for bit
against the CPU oracle: channel counts around the 16-byte quads and the
kernel's row sizes, and rows whose 3-sigma limits fall on or beside integers
(two-valued and near-constant rows), where the kernel has to follow the
reference's own rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NCHANS = [1, 5, 15, 16, 17, 31, 128, 1000, 1023, 1024, 1025, 2048, 3001, 4096, 4111, 8192, 8193]


def _rows(nchans, rng):
    """Rows of every kind, as uint8 [n, nchans]."""
    rows = []
    for d in (1, 2, 3, 4, 8, 16, 85):     # two values: mean -+ 3 sigma at or near integers
        for k in range(12):
            lo = int(rng.integers(0, 256 - d))
            r = np.where(rng.permutation(nchans) < max(1, nchans * (k + 1) // 24), lo + d, lo)
            rows.append(r)
            r = r.copy()                   # and a few channels around the limits
            n = min(nchans, 6)
            r[rng.permutation(nchans)[:n]] = np.clip(lo + d // 2 + 3 * d * np.array([-1, 1, -0.5, 0.5, 2, -2])[:n], 0, 255)
            rows.append(r)
    for sigma in (0.2, 0.6, 1.0, 3.0, 12.0, 40.0):
        for _ in range(10):
            r = np.clip(np.rint(rng.normal(rng.uniform(0, 255), sigma, nchans)), 0, 255)
            rows.append(r)
            r = r.copy()
            r[rng.random(nchans) < 0.05] = rng.integers(0, 256)
            rows.append(r)
    rows += [np.zeros(nchans), np.full(nchans, 255), rng.integers(0, 256, nchans), np.arange(nchans) % 256]
    one = np.zeros(nchans)
    one[-1] = 255
    rows.append(one)
    return np.stack(rows).astype(np.uint8)


@pytest.mark.parametrize("nchans", NCHANS)
def test_rows_match_oracle(aa, oracle, cuda, nchans):
    import torch
    print(f"outliers rows {nchans} channels", flush=True)
    rng = np.random.default_rng(nchans)
    x = _rows(nchans, rng)
    for nbits in (8, 4):
        y = x if nbits == 8 else (x >> 4)
        top = (1 << nbits) - 1
        bp = rng.uniform(0.3 * top, 0.7 * top, nchans).astype(np.float32)
        want = oracle.zero_dm_outliers(y, bandpass=bp, nbits=nbits)
        d = torch.from_numpy(np.concatenate([y, np.full((1, nchans), 7, np.uint8)])).to(cuda)
        aa.zero_dm_outliers(d[:-1], torch.from_numpy(bp).to(cuda), nbits=nbits)
        got = d.cpu().numpy()
        np.testing.assert_array_equal(got[:-1], want)
        assert np.all(got[-1] == 7)   # nothing written past the last row

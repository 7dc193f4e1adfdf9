"""GPU: the grouped maximum of the first single-pulse pass at W = 32 (the
widths are compared in fours, the winning four once more), on tiles where
every width fits, against the float64 oracle.  Tolerances as in
test_gpu_spd.py: the sums are the same float32 sums."""
import numpy as np
import pytest

from test_gpu_spd import check_first_pass

pytestmark = pytest.mark.gpu

TILE = 8192


@pytest.mark.parametrize("nsamp", [TILE + 31, TILE + 30, 2 * TILE + 32, 2 * TILE + 36])
@pytest.mark.parametrize("outputs", ["both", "snr", "width"])
def test_every_width_wins(aa, cuda, nsamp, outputs):
    """A pulse of each width 1..32 on its own row, at a tile's first samples,
    in the middle and across its end; rows of outputs at every alignment."""
    import torch
    rng = np.random.default_rng(nsamp)
    x = rng.normal(40.0, 1.0, size=(32, nsamp)).astype(np.float32)
    starts = [0, 4097, TILE - 17]
    for w in range(1, 33):
        for t in starts:
            x[w - 1, t:t + w] += 12.0 + 20.0 / w
    d = torch.zeros((32, nsamp + 3), dtype=torch.float32, device=cuda)
    d[:, :nsamp] = torch.from_numpy(x).to(cuda)
    msd = torch.empty((32, 2), dtype=torch.float32, device=cuda)
    snr = torch.full((32, nsamp + 1), -7.0, dtype=torch.float32, device=cuda)
    width = torch.full((32, nsamp + 1), -7, dtype=torch.int16, device=cuda)
    aa.spd_first_pass_raw(d.data_ptr(), d.stride(0), 32, nsamp, 32, msd, snr if outputs != "width" else None,
                          width if outputs != "snr" else None)
    both = aa.spd_first_pass(d[:, :nsamp], 32)
    torch.cuda.synchronize()
    check_first_pass(x, 32, both[0].cpu().numpy(), both[1].cpu().numpy(), both[2].cpu().numpy().astype(np.int64))
    assert sorted(both[2].unique().tolist()) == list(range(1, 33))
    assert torch.equal(msd, both[0])
    for got, want in ((snr, both[1]), (width, both[2])):
        if got is (snr if outputs == "width" else width if outputs == "snr" else None):
            assert bool((got == -7).all())
        else:
            assert torch.equal(got[:, :nsamp], want) and bool((got[:, nsamp:] == -7).all())


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_plane_that_is_not_finite(aa, cuda, bad):
    """One sample that is no number makes every mean one: SNR NaN, width 1."""
    import torch
    x = torch.randn((3, TILE + 100), device=cuda)
    x[1, 5000] = bad
    _, snr, width = aa.spd_first_pass(x, 32)
    assert bool(torch.isnan(snr).all()) and bool((width == 1).all())


def test_a_flat_plane(aa, cuda):
    """No spread: SNR 0 at every width, the smallest width wins."""
    import torch
    x = torch.full((3, TILE + 100), 3.0, device=cuda)
    msd, snr, width = aa.spd_first_pass(x, 32)
    assert bool((msd[:, 1] == 0).all())
    assert bool((snr == 0).all()) and bool((width == 1).all())


@pytest.mark.parametrize("W", [1, 2, 5, 7, 8, 9, 15, 16, 17, 31])
@pytest.mark.parametrize("nsamp", ["all widths of one tile", "one short", "two tiles and 8", "two tiles and 31"])
def test_other_width_limits(aa, cuda, W, nsamp):
    """Limits between the 8, 16 and 32 the kernels are compiled for."""
    import torch
    n = {"all widths of one tile": TILE + W - 1, "one short": TILE + max(W - 2, 0), "two tiles and 8": 2 * TILE + 8,
         "two tiles and 31": 2 * TILE + 31}[nsamp]
    rng = np.random.default_rng(100 * W + n)
    x = rng.normal(40.0, 1.0, size=(5, n)).astype(np.float32)
    x[3, 4000:4000 + W] += 9.0
    x[4, TILE - 3:TILE - 3 + W] += 9.0
    msd, snr, width = aa.spd_first_pass(torch.from_numpy(x).to(cuda), W)
    check_first_pass(x, W, msd.cpu().numpy(), snr.cpu().numpy(), width.cpu().numpy().astype(np.int64))
    x[1, 77] = np.nan
    _, snr, width = aa.spd_first_pass(torch.from_numpy(x).to(cuda), W)
    assert bool(torch.isnan(snr).all()) and bool((width == 1).all())

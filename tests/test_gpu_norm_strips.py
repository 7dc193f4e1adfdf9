"""GPU: column normalisation at the edges of its row counts, strips, segments
and lane numbering, bit for bit against the oracle (the float sums keep the
oracle's order, so there is no tolerance)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ndms, nsamp: the row limits of each register size, the last kernel beyond
# them, and strips of 64 columns with every remainder
PLANES = [(r, c) for r, c in [(1, 64), (31, 3), (32, 128), (33, 65), (128, 66), (129, 127), (256, 191), (257, 64),
                              (512, 130), (513, 61), (1024, 190), (1025, 129), (1535, 63), (1536, 257), (1537, 70),
                              (65, 4095), (65, 4096), (1100, 4131), (700, 16391),
                              (1537, 40960), (1601, 41003), (4, 40964)]]   # 4 columns per lane, where words are aligned


@pytest.mark.parametrize("ndms,nsamp", PLANES)
@pytest.mark.parametrize("offset", [0, 1])
def test_output_planes(aa, oracle, cuda, ndms, nsamp, offset):
    import torch
    rng = np.random.default_rng(ndms * 31 + nsamp)
    plane = rng.normal(127.0, 30.0, size=(ndms, nsamp)).astype(np.float32)
    plane[0, :] += 1.0e6   # the order of the sums shows
    flat = torch.full((offset + ndms * nsamp + 4,), -3.0, dtype=torch.float32, device=cuda)
    d = flat[offset:offset + ndms * nsamp].view(ndms, nsamp)
    d.copy_(torch.from_numpy(plane))
    aa.output_ddtr_normalization(d)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(d.cpu().numpy(), oracle.output_normalization(plane))
    assert bool((flat[:offset] == -3.0).all()) and bool((flat[offset + ndms * nsamp:] == -3.0).all())


@pytest.mark.parametrize("nsamp,nchans", [(31, 16), (33, 48), (512, 16), (513, 400), (8192, 32), (8193, 32),
                                          (20001, 16), (4097, 1040),
                                          (1, 1), (31, 1), (33, 7), (1000, 3), (777, 99), (2049, 130), (8223, 257)])
@pytest.mark.parametrize("fill", ["noise", "full"])
@pytest.mark.parametrize("offset", [0, 4, 3])
def test_input_rows(aa, oracle, cuda, nsamp, nchans, fill, offset):
    """u8: lanes numbered through the bytes of 32 rows, two columns to a 32-bit
    sum (full: the largest sums), at word and odd byte addresses."""
    import torch
    rng = np.random.default_rng(nsamp + nchans)
    x = rng.integers(0, 256, size=(nsamp, nchans), dtype=np.uint8)
    if fill == "full":
        x[:, ::3] = 255
    flat = torch.full((offset + nsamp * nchans + 16,), 77, dtype=torch.uint8, device=cuda)
    d = flat[offset:offset + nsamp * nchans].view(nsamp, nchans)
    d.copy_(torch.from_numpy(x))
    aa.input_ddtr_normalization(d)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(d.cpu().numpy(), oracle.input_normalization(x))
    assert bool((flat[:offset] == 77).all()) and bool((flat[offset + nsamp * nchans:] == 77).all())

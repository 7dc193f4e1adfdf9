"""aa_hip_host_copy (CPU): every byte and no other, at one thread's sizes, at
the thread counts' edges and at odd addresses."""
import ctypes

import numpy as np
import pytest

MIB = 1 << 20


@pytest.mark.parametrize("bytes_", [0, 1, 4095, 8 * MIB - 1, 8 * MIB, 8 * MIB + 1, 12 * MIB + 4097, 33 * MIB + 5])
@pytest.mark.parametrize("offset", [0, 3])
def test_host_copy(aa, bytes_, offset):
    lib = aa.load_library()
    src = np.random.default_rng(bytes_).integers(0, 256, size=bytes_ + offset + 8, dtype=np.uint8)
    dst = np.full(bytes_ + offset + 8, 0x5A, dtype=np.uint8)
    assert lib.aa_hip_host_copy(dst.ctypes.data + offset, src.ctypes.data + offset, bytes_) == 0
    np.testing.assert_array_equal(dst[offset:offset + bytes_], src[offset:offset + bytes_])
    assert np.all(dst[:offset] == 0x5A) and np.all(dst[offset + bytes_:] == 0x5A)


def test_host_copy_refuses_null(aa):
    lib = aa.load_library()
    buf = ctypes.create_string_buffer(4)
    assert lib.aa_hip_host_copy(None, ctypes.addressof(buf), 4) != 0
    assert lib.aa_hip_host_copy(ctypes.addressof(buf), None, 4) != 0
    assert lib.aa_hip_host_copy(None, None, 0) == 0

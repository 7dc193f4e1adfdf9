"""aa_hip_host_copy (CPU): every byte and no other, at one thread's sizes, at
the thread counts' edges and at odd addresses."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import host_library  # noqa: E402

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


def test_host_copy_without_memory_for_threads(tmp_path):
    """Where a thread cannot be made the calling thread copies its part."""
    host_library.run('''
lib = aa.load_library()
src = np.random.default_rng(1).integers(0, 256, size=40 << 20, dtype=np.uint8)
dst = np.zeros_like(src)
fake.lib.fake_fail_host_allocations(1)
status = lib.aa_hip_host_copy(dst.ctypes.data, src.ctypes.data, src.nbytes)
fake.lib.fake_fail_host_allocations(2 ** 64 - 1)
assert status == 0 and np.array_equal(dst, src)
''', tmp_path)

"""Dedispersion routes without the memory for their tables: the range falls
back to the kernel it would have otherwise (CPU: the library's host code on a
HIP runtime without a GPU)."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import host_library  # noqa: E402

GEOMETRY = '''
import ddtr_oracle as oracle
ds = oracle.dmshifts(1024, 1500.0, -0.3)
tp, maxshift = 60000, 3000
def make(bits):
    return aa.DdtrPlan(ds, [(0.0, 0.5, 256, 1)], 64e-6, maxshift, tp, sample_bits=bits)
x, out = Tensor((tp + maxshift, 1024), 2), Tensor((256, tp))
'''


@pytest.mark.parametrize("which", [0, 1, 2, 3], ids=["tables", "flags", "planes", "sums"])
def test_16_bit_plan_without_memory(tmp_path, which):
    """Without any one of the matrix kernel's allocations a 16-bit range runs
    dedisperse_u16, with no error left behind and no table kept for nothing."""
    host_library.run(GEOMETRY + f'''
plan = make(16)
created = len(fake.allocations())
plan.execute_chunk(x, [tp], [out])
assert fake.ran("dedisperse_matrix_kernel")
sizes = fake.allocations()[created:]
assert len(sizes) == 4 and len(set(sizes)) == 4, sizes   # tables, flags, planes, sampled sums
plan.close()
plan = make(16)
blocks, bytes_ = fake.lib.fake_blocks(), fake.lib.fake_device_bytes()
assert plan.device_bytes() == bytes_
fake.fail_allocations(sizes[{which}], sizes[{which}] + 1)
for chunk in range(2):
    plan.execute_chunk(x, [tp], [out])
    names = fake.kernels()
    assert any("dedisperse_u16_kernel" in n for n in names) and not any("matrix" in n for n in names), names
    fake.fail_allocations()   # the choice stays what it was on the first chunk
assert fake.lib.fake_blocks() == blocks and fake.lib.fake_device_bytes() == bytes_
assert plan.device_bytes() == bytes_
plan.close()
assert fake.lib.fake_device_bytes() == 0
''', tmp_path)


@pytest.mark.parametrize("where", ["device", "host"])
def test_8_bit_plan_without_memory(tmp_path, where):
    """Without the memory for the matrix kernel's tables an 8-bit range runs the
    LDS shape that fits, from its first call on."""
    host_library.run(GEOMETRY + f'''
x = Tensor((tp + maxshift, 1024), 1)
plan = make(8)
created = len(fake.allocations())
plan.execute_chunk(x, [tp], [out])
assert fake.ran("dedisperse_matrix_kernel")
tables, = fake.allocations()[created:]
plan.close()
plan = make(8)
plan.ingest(x, tp)
if "{where}" == "device":
    fake.fail_allocations(tables, tables + 1)
else:
    fake.lib.fake_fail_host_allocations(tables)   # the tables are put together in host memory
plan.run_range(0, tp, out)
names = fake.kernels()
assert any("dedisperse_wide_kernel" in n for n in names) and not any("matrix" in n for n in names), names
fake.fail_allocations()
fake.lib.fake_fail_host_allocations(2 ** 64 - 1)
plan.run_range(0, tp, out)
assert not fake.ran("matrix")
assert plan.device_bytes() == fake.lib.fake_device_bytes()
''', tmp_path)

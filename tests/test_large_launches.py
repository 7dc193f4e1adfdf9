"""Calls of more work-groups than one launch takes along x (2^32 threads), on the
CPU: the library's host code on a HIP runtime without a GPU."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import host_library  # noqa: E402


def test_rows(tmp_path):
    """17 million work-groups of the row kernel: a range whose trials are too far
    apart for any shape, a plane of 69 GB."""
    host_library.run('''
import ddtr_oracle as oracle
ds = oracle.dmshifts(2, 1500.0, -100.0)
ndms, tp, step = 16500, 1 << 20, 60.0
shift = int(ds[-1] * step * ndms / 64e-6) + 10
plan = aa.DdtrPlan(ds, [(0.0, step, ndms, 1)], 64e-6, shift, tp)
plan.ingest(Tensor((tp + shift, 2), 1), tp)
out = Tensor((1, tp))     # never written: no kernel runs
fake.kernels()
plan.run_range(0, tp, out)
names = fake.kernels()
assert len(names) == 1 and "dedisperse_rows_kernel" in names[0], names
''', tmp_path)

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


def test_output_normalisation_of_a_long_plane(tmp_path):
    """600 million columns."""
    host_library.run('''
fake.kernels()
for rows in (3, 2000):
    aa.check(aa.load_library().aa_hip_output_ddtr_normalization(Tensor((1, 1)).data_ptr(), rows, 600000001, None))
    assert len(fake.kernels()) == 1
''', tmp_path)


def test_refinement_of_many_windows(tmp_path):
    """Five million windows of one channel and eight samples, energy loss."""
    host_library.run('''
n = 5000000
lib = aa.load_library()
i64, i32 = ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_int)
xo, do = np.arange(n, dtype=np.int64) * 8, np.zeros(n, dtype=np.int64)
nc, ns = np.full(n, 1, dtype=np.int32), np.full(n, 8, dtype=np.int32)
h = ctypes.c_void_p()
aa.check(lib.aa_hip_refine_create(0, n, xo.ctypes.data_as(i64), do.ctypes.data_as(i64), nc.ctypes.data_as(i32),
                                  ns.ctypes.data_as(i32), ctypes.byref(h)))
p = Tensor((1, 1)).data_ptr()   # never read: no kernel runs
fake.kernels()
aa.check(lib.aa_hip_refine_run(h, p, p, p, p, p, p, p, 3, -1.0, 0.5, 2, 0.5, 1e-4, None))
assert len(fake.kernels()) == 3 + 2 * 3      # a scan pass and three evaluations
''', tmp_path)

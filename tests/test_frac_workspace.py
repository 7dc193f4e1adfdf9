"""Scratch memory of a FracPlan's calls (CPU: the library's host code on a HIP
runtime without a GPU)."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import host_library  # noqa: E402

PLAN = '''
import frac_ddtr
import torch
C, T, K, B = 1024, 256, 16, 2
plan = frac_ddtr.FracPlan(np.linspace(0, 3, C).astype(np.float32), np.linspace(-1, 1, K).astype(np.float32), T, B)
x, y, dm = Tensor((B, C, T)), Tensor((B, K, T)), Tensor((B,))
Y_PART, GDM_PART = 13, 4   # words of frac_args
'''


def test_plan_without_memory_for_partial_profiles(tmp_path):
    """The C calls without a workspace argument use the plan's: without the
    memory for the partial profiles the plan is made all the same and its
    forward calls are not split."""
    host_library.run(PLAN + '''
lib = aa.load_library()
largest = max(fake.allocations())
fake.fail_allocations(largest, largest + 1)
plan = frac_ddtr.FracPlan(plan.delay_per_dm, plan.trials, T, B)
args = (plan.handle, x.data_ptr(), B, dm.data_ptr(), y.data_ptr())
fake.kernels()
aa.check(lib.aa_hip_frac_forward(*args, None))
names = fake.kernels()
assert len(names) == 1 and "frac_rows_kernel" in names[0], names
''', tmp_path)

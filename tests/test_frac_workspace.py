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


def test_calls_share_no_scratch(tmp_path):
    """Two forward calls, or two gradients, of one plan may run on two streams at
    once: each has partial sums of its own, in memory of its stream."""
    host_library.run(PLAN + '''
kept = []
empty = torch.empty
torch.empty = lambda *a, **k: kept.append(empty(*a, **k)) or kept[-1]
for handle in (4096, 8192):
    torch.cuda.current_stream = lambda *a, handle=handle: Stream(handle)
    plan.forward(x, dm)
    plan.adjoint(x, y, dm)
forward = fake.argument_words("frac_rows_kernelILi2ELb0E", Y_PART) + fake.argument_words("frac_rows_kernelILi1ELb0E", Y_PART)
adjoint = fake.argument_words("frac_rows_kernelILi2ELb1E", GDM_PART) + fake.argument_words("frac_rows_kernelILi1ELb1E", GDM_PART)
assert len(forward) == len(adjoint) == 2
assert fake.ran("frac_sum_parts_kernel")       # the channels are split
assert all(forward) and len(set(forward)) == 2 and len(set(adjoint)) == 2
assert set(forward + adjoint) <= {t.data_ptr() for t in kept}
''', tmp_path)


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
forward, adjoint = ctypes.c_size_t(), ctypes.c_size_t()
aa.check(lib.aa_hip_frac_workspace_bytes(plan.handle, B, ctypes.byref(forward), ctypes.byref(adjoint)))
work = Tensor((forward.value,), 1)
assert lib.aa_hip_frac_forward_ws(*args, work.data_ptr(), forward.value - 1, None) == aa.AA_HIP_ERROR_INVALID_ARGUMENT
aa.check(lib.aa_hip_frac_forward_ws(*args, work.data_ptr(), forward.value, None))
assert fake.ran("frac_sum_parts_kernel")
gx, gdm = Tensor((B, C, T)), Tensor((B,), 8)
args = (plan.handle, x.data_ptr(), y.data_ptr(), B, dm.data_ptr(), gx.data_ptr(), gdm.data_ptr())
assert lib.aa_hip_frac_adjoint_ws(*args, work.data_ptr(), adjoint.value - 1, None) == aa.AA_HIP_ERROR_INVALID_ARGUMENT
aa.check(lib.aa_hip_frac_adjoint_ws(*args, work.data_ptr(), adjoint.value, None))
aa.check(lib.aa_hip_frac_adjoint_ws(*args[:6], None, None, 0, None))     # without the DMs' gradient: no scratch
''', tmp_path)

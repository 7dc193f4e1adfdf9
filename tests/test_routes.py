"""Which kernel a range's call launches (CPU: the library's host code on a HIP
runtime without a GPU)."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import host_library  # noqa: E402

GEOMETRY = '''
import ddtr_oracle as oracle
ds = oracle.dmshifts(1024, 1500.0, -0.3)
tp, maxshift = 60000, 3000
x, out = Tensor((tp + maxshift, 1024), 1), Tensor((256, tp))
def make(bits=8, nranges=1):
    return aa.DdtrPlan(ds, [(0.0, 0.5, 256, 1)] * nranges, 64e-6, maxshift, tp, sample_bits=bits)
'''


def test_forced_lds_kernel_is_the_lds_kernel(tmp_path):
    """AA_HIP_KERNEL_LDS on a handle, alone and in a batch, runs the first LDS
    shape that fits, as the handle-free call does; AA_HIP_KERNEL_MATRIX the
    matrix kernel, or nothing where it does not take the range."""
    host_library.run(GEOMETRY + '''
plan = make()
plan.ingest(x, tp)
plan.run_range(0, tp, out)
assert fake.ran("dedisperse_matrix_kernel")
plan.set_kernel(aa.KERNEL_LDS)
plan.run_range(0, tp, out)
assert fake.ran("dedisperse_wide_kernel")
batch = aa.DdtrBatch([plan])
batch.execute([x], [[tp]], [[out]], use_graph=False)
names = fake.kernels()
assert any("dedisperse_wide_batch_kernel" in n for n in names) and not any("matrix" in n for n in names), names
plan.set_kernel(aa.KERNEL_MATRIX)
plan.run_range(0, 600, out)      # small: the automatic choice would be the rows
assert fake.ran("dedisperse_matrix_kernel")
plan.set_kernel(aa.KERNEL_AUTO)
plan.run_range(0, 600, out)
assert fake.ran("dedisperse_rows_kernel")
coarse = aa.DdtrPlan(ds, [(0.0, 40.0, 64, 1)], 64e-6, maxshift * 20, tp)
xc = Tensor((tp + maxshift * 20, 1024), 1)
coarse.set_kernel(aa.KERNEL_MATRIX)
coarse.ingest(xc, tp)
try:
    coarse.run_range(0, tp, out)
    raise SystemExit("the matrix kernel does not take this range")
except aa.AAHipError as e:
    assert e.status == aa.AA_HIP_ERROR_UNSUPPORTED
try:
    aa.dedisperse_u8(x, 63232, 63000, ds, x, 256, tp, 0.0, 1.0, 1, out, tp, kernel=aa.KERNEL_MATRIX)
    raise SystemExit("the handle-free call has no matrix kernel")
except aa.AAHipError as e:
    assert e.status == aa.AA_HIP_ERROR_INVALID_ARGUMENT
''', tmp_path)


TUNING = GEOMETRY + '''
import json
import multibeam as mb

class Strategy:
    def dm(self, r):
        return (0.0, 128.0, 0.5, 1, 1)

def beam(plan, n=1):
    return mb.Beam(dict(nchans=1024), Strategy(), plan, x, [out] * n, [tp] * n, [256] * n)

def kernel_alone(plan):
    plan.ingest(x, tp)
    fake.kernels()
    plan.run_range(0, tp, out)
    return fake.kernels()

def kernel_batched(plans, tp=tp):
    batch = aa.DdtrBatch(plans)
    batch.execute([x] * len(plans), [[tp]] * len(plans), [[out]] * len(plans), use_graph=False)
    return [n for n in fake.kernels() if "dedisperse" in n]
'''


def test_captured_tables_outlive_a_change_of_shape(tmp_path):
    """A captured batch reads the plan tables of its ranges' shapes: another
    shape's call on the handle, or autotuning it, leaves them in place."""
    host_library.run(TUNING + '''
plan = make()
plan.set_range_variant(0, 4)
batch = aa.DdtrBatch([plan])
batch.execute([x], [[tp]], [[out]], use_graph=True)
captured = set(fake.blocks())
for variant in (5, 6, 4, 2):
    plan.set_range_variant(0, variant)
    plan.run_range(0, tp, out)
    assert captured <= set(fake.blocks()), variant
had = len(fake.blocks())
plan.autotune_range(0, tp, out, 1)
assert captured <= set(fake.blocks())
assert len(fake.blocks()) <= had + 2          # keeps the best shape's and the automatic choice's, no others
plan.close()
''', tmp_path)


def test_autotuned_class_runs_one_kernel(tmp_path):
    """Two beams of one class, and a third from the reloaded cache, keep what
    the autotuner found fastest: here the matrix kernel."""
    cache = tmp_path / "tune.json"
    host_library.run(TUNING + f'''
path = {str(cache)!r}
fake.lib.fake_cost(b"dedisperse_matrix", 0.5)
fake.lib.fake_cost(b"dedisperse_wide_kernelILi4ELi3E", 0.7)   # shape 5; the other shapes take 1 ms
a, b, c = make(), make(), make()
mb.autotune([beam(a), beam(b)], cache_path=path)
mb.autotune([beam(c)], cache_path=path)
for plan in (a, b, c):
    assert plan.range_tuning(0) == (5, True)
    assert any("dedisperse_matrix_kernel" in n for n in kernel_alone(plan))
names = kernel_batched([a, b, c])
assert len(names) == 3 and all("dedisperse_matrix_kernel" in n for n in names), names
# in a batch a range too small for a matrix launch of its own takes the shape that was fastest
names = kernel_batched([a, b, c], 9000)
assert len(names) == 1 and "dedisperse_wide_batch_kernelILi4ELi3E" in names[0], names
''', tmp_path)


def test_autotuned_class_on_an_lds_shape(tmp_path):
    """The same where a shape is fastest; and a cache file without the automatic
    choice's time is timed again."""
    cache = tmp_path / "tune.json"
    host_library.run(TUNING + f'''
path = {str(cache)!r}
fake.lib.fake_cost(b"dedisperse_wide_kernelILi4ELi3E", 0.3)
a, b, c = make(), make(), make()
mb.autotune([beam(a), beam(b)], cache_path=path)
mb.autotune([beam(c)], cache_path=path)
for plan in (a, b, c):
    assert plan.range_tuning(0) == (5, False)
    assert any("dedisperse_wide_kernelILi4ELi3E" in n for n in kernel_alone(plan))
old = json.load(open(path))
for v in old.values():
    del v["automatic"]
json.dump(old, open(path, "w"))
fake.lib.fake_cost(b"dedisperse_matrix", 0.2)
d = make()
mb.autotune([beam(d)], cache_path=path)
assert d.range_tuning(0) == (5, True)
assert all(v["automatic"] for v in json.load(open(path)).values())
''', tmp_path)


CAPTURE = GEOMETRY + '''
capture = Stream(4096)
def captured(call):
    """The kernels of a call under capture, which it must not break."""
    fake.kernels()
    fake.lib.fake_capture(4096)
    call()
    broken = fake.lib.fake_capture_broken()
    fake.lib.fake_capture(None)
    assert not broken, "the call allocated or synchronised under capture"
    return fake.kernels()
'''


def test_16_bit_chunk_captured_at_first(tmp_path):
    """A 16-bit chunk may be captured without an eager call before it: what the
    matrix kernel needs is not there, so dedisperse_u16 runs; eager calls and
    captures after one take the matrix kernel."""
    host_library.run(CAPTURE + '''
maxshift *= 3
x16, half = Tensor((tp + maxshift, 1024), 2), tp // 2
plan = aa.DdtrPlan(ds, [(0.0, 0.5, 256, 1), (128.0, 1.0, 128, 2)], 64e-6, maxshift, tp, sample_bits=16)
outs = [out, Tensor((128, half))]
def chunk():
    plan.execute_chunk(x16, [tp, half], outs, stream=capture)
names = captured(chunk)
assert sum("dedisperse_u16_kernel" in n for n in names) == 2 and not any("matrix" in n for n in names), names
# eager up to the first range: the second one's level has no planes yet
plan.ingest(x16, tp)
plan.run_range(0, tp, out)
assert fake.ran("dedisperse_matrix_kernel")
names = captured(lambda: plan.run_range(1, half, outs[1], stream=capture))
assert any("dedisperse_u16_kernel" in n for n in names) and not any("matrix" in n for n in names), names
chunk()
assert sum("dedisperse_matrix_kernel" in n for n in fake.kernels()) == 2
assert sum("dedisperse_matrix_kernel" in n for n in captured(chunk)) == 2
''', tmp_path)


def test_captured_chunk_longer_than_the_eager_one(tmp_path):
    """A short eager chunk goes from the rows, and so does a longer one captured
    after it, whose shape's tables are not there; after an eager one it takes
    the shape."""
    host_library.run(CAPTURE + '''
ds = oracle.dmshifts(128, 1500.0, -5.0)   # a range that the matrix kernel does not take
shift = int(ds[-1] * 256.0 / 64e-6) + 10
plan = aa.DdtrPlan(ds, [(0.0, 0.5, 512, 1)], 64e-6, shift, tp)
xl, ol = Tensor((tp + shift, 128), 1), Tensor((512, tp))
plan.ingest(xl, 100)
plan.run_range(0, 100, ol)
assert fake.ran("dedisperse_rows_kernel")
plan.ingest(xl, tp)
def chunk():
    plan.run_range(0, tp, ol, stream=capture)
assert any("dedisperse_rows_kernel" in n for n in captured(chunk))
chunk()
assert fake.ran("dedisperse_wide_kernel")
assert any("dedisperse_wide_kernel" in n for n in captured(chunk))
''', tmp_path)


def test_8_bit_range_captured_at_first(tmp_path):
    """A range left to the automatic choice may be captured at once: it goes from
    the rows or on a shape that reads no tables."""
    host_library.run(CAPTURE + '''
plan = make()
plan.ingest(x, tp)
assert any("dedisperse_rows_kernel" in n for n in captured(lambda: plan.run_range(0, tp, out, stream=capture)))
plan.set_range_tuning(0, 0, True)
names = captured(lambda: plan.run_range(0, tp, out, stream=capture))
assert any("dedisperse_lds_kernel" in n or "dedisperse_rows_kernel" in n for n in names), names
plan.run_range(0, tp, out)
assert fake.ran("dedisperse_matrix_kernel")
''', tmp_path)


def test_output_normalisation_of_tall_planes(tmp_path):
    """Planes of more rows than a strip keeps in registers, or of next to none: 4
    columns per lane where the plane is wide and its words are aligned."""
    host_library.run('''
plane = Tensor((1, 1)).data_ptr()
def kernel(rows, cols, at=plane):
    fake.kernels()
    aa.check(aa.load_library().aa_hip_output_ddtr_normalization(at, rows, cols, None))
    return fake.kernels()[0]
assert "normalize_strip_f32_kernel" in kernel(1536, 222656)
assert "normalize_strip_f32_kernel" in kernel(5, 222656)
assert "normalize_strip_f32_kernel" in kernel(4, 222657)
assert "normalize_strip_f32_kernel" in kernel(4, 4096)
assert "normalize_columns_f32x4_kernel" in kernel(4, 222656)
assert "normalize_columns_f32x4_kernel" in kernel(1537, 222656)
assert "normalize_columns_f32x4_kernel" in kernel(6080, 40960)
for rows, cols, at in ((6080, 40956, plane), (1537, 222657, plane), (1537, 222656, plane + 4)):
    assert "normalize_columns_kernel" in kernel(rows, cols, at)
''', tmp_path)


def test_level_0_of_unaligned_rows(tmp_path):
    """The wide corner turn where it has tiles enough; the byte kernel for less,
    and the wide one at any size where binned levels follow or rows are aligned."""
    host_library.run('''
at = Tensor((1, 1)).data_ptr()
def kernel(nsamp, nchans, levels=1):
    fake.kernels()
    pitch = (nsamp + 255) // 256 * 256
    aa.corner_turn_levels(Tensor((1, 1)), 1, nsamp, nchans, [Tensor((1, 1))] * levels, [pitch] * levels)
    return fake.kernels()[0]
for nsamp, nchans in ((500, 2001), (4000, 1000), (100000, 40), (24000, 200), (8000, 1000)):
    assert "18corner_turn_kernel" in kernel(nsamp, nchans), (nsamp, nchans)
for nsamp, nchans in ((24000, 500), (100000, 65), (4000, 4097), (500, 2000), (200, 16)):
    assert "corner_turn_wide_kernel" in kernel(nsamp, nchans), (nsamp, nchans)
ds = np.linspace(0, 1e-3, 99).astype(np.float32)
plan = aa.DdtrPlan(ds, [(0.0, 0.5, 16, 1), (8.0, 1.0, 16, 2)], 64e-6, 400, 1400)
fake.kernels()
plan.ingest(Tensor((1800, 99), 1), 1400)
assert fake.ran("corner_turn_wide_kernel")
''', tmp_path)


def test_refinement_items(tmp_path):
    """Few windows are split into smaller items; many keep 256 channels each."""
    host_library.run('''
import frac_ddtr
def items(n, C, T):
    plan = frac_ddtr.RefinePlan([C] * n, [T] * n, [0] * n, [0] * n, loss="energy")
    p, h = Tensor((1, 1)).data_ptr(), plan.handle
    fake.kernels()
    aa.check(aa.load_library().aa_hip_refine_run(h, p, p, p, p, p, p, p, 0, 0.0, 0.0, 0, 0.5, 1e-4, None))
    return [fake.lib.fake_launch_grid(i) for i in range(fake.lib.fake_launches())
            if b"refine_partial" in fake.lib.fake_launch_name(i)][0]
assert items(1, 64, 64) == 4
assert items(32, 256, 256) == 32 * 16
assert items(64, 256, 256) == 64 * 16
assert items(256, 256, 256) == 256 * 4
assert items(1, 4096, 1024) == 64
assert items(16, 4096, 2048) == 16 * 2 * 32
assert items(100, 4096, 1024) == 100 * 16
assert items(5000, 16, 2000) == 5000 * 2
''', tmp_path)


def test_16_bit_ranges_on_the_faster_kernel(tmp_path):
    """Few channels, or trials far apart, keep dedisperse_u16, and no byte planes
    are made for them."""
    host_library.run('''
import ddtr_oracle as oracle
def kernels(nchans, ndms, tp, step, kernel=0):
    ds = oracle.dmshifts(nchans, 1500.0, -300.0 / nchans)
    shift = int(ds[-1] * step * ndms / 64e-6) + 16
    plan = aa.DdtrPlan(ds, [(0.0, step, ndms, 1)], 64e-6, shift, tp, sample_bits=16)
    plan.set_kernel(kernel)
    fake.kernels()
    plan.execute_chunk(Tensor((tp + shift, nchans), 2), [tp], [Tensor((ndms, tp))])
    return " ".join(fake.kernels())
for case in ((16, 64, 4000, 0.5), (40, 1000, 200000, 2.0), (56, 64, 16000, 2.0), (32, 16, 200, 0.5)):
    names = kernels(*case)
    assert "dedisperse_u16_kernel" in names and "matrix" not in names and "split_u16" not in names, case
for case in ((40, 256, 60000, 0.25), (64, 64, 60000, 0.25), (128, 16, 1000, 0.5), (1024, 256, 60000, 0.5)):
    assert "dedisperse_matrix_kernel" in kernels(*case), case
assert "dedisperse_matrix_kernel" in kernels(16, 64, 4000, 0.5, aa.KERNEL_MATRIX)
''', tmp_path)


def test_matrix_launches_in_a_batch(tmp_path):
    """Ranges of many tiles take matrix launches of their own in a batch where
    that is faster than the shared launch: not with few channels."""
    host_library.run('''
import ddtr_oracle as oracle
def ran(nchans, ndms, tp, step, band, fch1):
    ds = oracle.dmshifts(nchans, fch1, -band / nchans)
    shift = int(ds[-1] * step * ndms / 64e-6) + 16
    plan = aa.DdtrPlan(ds, [(0.0, step, ndms, 1)], 64e-6, shift, tp)
    batch = aa.DdtrBatch([plan])
    batch.execute([Tensor((tp + shift, nchans), 1)], [[tp]], [[Tensor((ndms, tp))]], use_graph=False)
    return plan.range_kernel(0)
for case in ((64, 512, 30000, 0.25, 300.0, 1500.0), (192, 512, 30000, 0.5, 810.0, 1760.0),
             (256, 128, 120000, 0.5, 810.0, 1760.0), (64, 128, 120000, 0.25, 300.0, 1500.0)):
    assert 0 <= ran(*case) < aa.LDS_SHAPES, case
for case in ((1024, 512, 30000, 0.25, 300.0, 1500.0), (512, 256, 60000, 0.25, 300.0, 1500.0),
             (1024, 1000, 60000, 0.5, 810.0, 1760.0), (128, 1000, 60000, 0.25, 300.0, 1500.0)):
    assert ran(*case) == aa.RANGE_MATRIX, case
''', tmp_path)

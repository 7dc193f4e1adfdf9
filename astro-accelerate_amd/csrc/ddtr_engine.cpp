// Dedispersion engine: corner turn -> x2 cascade -> per-range dedispersion,
// all on caller streams, with every launch validated on the host first.
#include "ddtr_engine.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>

#include "aa_ddtr_hip.h"
#include "ddtr_lds.h"

namespace aa_hip {

namespace {
thread_local std::string g_last_error;

size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

int fail(int code, const std::string &msg) {
    set_last_error(msg);
    return code;
}

int hip_fail(hipError_t e, const char *what) {
    return fail(e == hipErrorOutOfMemory ? AA_HIP_ERROR_OUT_OF_MEMORY : AA_HIP_ERROR_DEVICE,
                std::string(what) + ": " + hipGetErrorString(e));
}

// Whether s is being captured into a graph, or cannot be asked because another
// stream is: allocations and synchronous copies would break the capture.
bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

int no_matrix() {
    return fail(AA_HIP_ERROR_UNSUPPORTED, "the matrix kernel does not take this range (its plan does not fit or does "
                                          "not pay, or there is no memory for its tables)");
}

// A batched range with this many tiles fills the GPU's 256 work-groups twice
// over and may run a matrix launch of its own (matrix_beats_shared); smaller ones
// stay in the shared launches (96 beams of 64-256 channels: 1.98 ms batched, 4.27
// ms with a matrix launch per range).
constexpr long kMatrixAloneTiles = 512;

bool is_pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }
int log2i(int v) {
    int k = 0;
    while ((1 << k) < v) ++k;
    return k;
}

struct device_guard {
    int prev = -1;
    explicit device_guard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        if (prev != dev) (void)hipSetDevice(dev);
    }
    ~device_guard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};
}  // namespace

void set_last_error(const std::string &msg) { g_last_error = msg; }
const char *last_error() { return g_last_error.c_str(); }

int check_delays(const float *dmshifts, int nchans, int ndms, float mstartdm, float mdmstep,
                 int t_processed, long row_len) {
    if (ndms <= 0 || t_processed <= 0) return AA_HIP_SUCCESS;
    // delay(c, d) is monotone in d for each c (fma of a non-negative step),
    // so the extremes over d are at d = 0 and d = ndms - 1.
    long lo = 0, hi = 0;
    for (int c = 0; c < nchans; ++c) {
        const long a = host_delay(dmshifts[c], 0, mstartdm, mdmstep);
        const long b = host_delay(dmshifts[c], ndms - 1, mstartdm, mdmstep);
        lo = std::min(lo, std::min(a, b));
        hi = std::max(hi, std::max(a, b));
    }
    if (lo < 0)
        return fail(AA_HIP_ERROR_UNSUPPORTED,
                    "negative dispersion delay (ascending channel frequencies are not supported)");
    if ((long)t_processed + hi > row_len)
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT,
                    "rows too short: t_processed " + std::to_string(t_processed) + " + max delay " +
                        std::to_string(hi) + " > row length " + std::to_string(row_len));
    if (mdmstep < 0.0f) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "negative DM step");
    return AA_HIP_SUCCESS;
}

lds_choice choose_lds(const float *h_dmshifts, int nchans, int ndms, float mstartdm, float mdmstep, int variant) {
    lds_choice c{-1, -1};
    static const int order[kLdsVariants] = {4, 5, 2, 3, 0, 1, 6};
    for (int v : order) {
        if (variant >= 0 && v != variant) continue;
        const int q = lds_row_quads(v, h_dmshifts, nchans, ndms, mstartdm, mdmstep);
        if (q > 0) {
            c.variant = v;
            c.row_quads = q;
            return c;
        }
    }
    return c;
}

int resolve_launch(int kernel, const uint8_t *L, size_t pitch, int nchans, const float *d_dmshifts,
                   const float *h_dmshifts, int ndms, int t_processed, float mstartdm, float mdmstep, int inBin,
                   float *out, size_t out_pitch, lds_choice choice, range_launch *rl) {
    *rl = range_launch{};
    rl->L = L;
    rl->pitch = pitch;
    rl->nchans = nchans;
    rl->d_dmshifts = d_dmshifts;
    rl->ndms = ndms;
    rl->t_processed = t_processed;
    rl->mstartdm = mstartdm;
    rl->mdmstep = mdmstep;
    rl->inBin = inBin;
    rl->out = out;
    rl->out_pitch = out_pitch;
    rl->variant = -1;
    const int forced = kernel == AA_HIP_KERNEL_LDS_C32    ? 0
                       : kernel == AA_HIP_KERNEL_LDS_C16  ? 1
                       : kernel == AA_HIP_KERNEL_LDS_PAIR ? 4   // the widest pair tile that fits: 4, 5, 2
                       : kernel == AA_HIP_KERNEL_LDS_QUAD ? 3
                                                          : -1;
    if (kernel != AA_HIP_KERNEL_DIRECT && (pitch % 16) == 0 && ((uintptr_t)L % 16) == 0) {
        if (forced >= 0) {
            choice = choose_lds(h_dmshifts, nchans, ndms, mstartdm, mdmstep, forced);
            if (choice.variant < 0 && forced == 4) choice = choose_lds(h_dmshifts, nchans, ndms, mstartdm, mdmstep, 5);
            if (choice.variant < 0 && forced == 4) choice = choose_lds(h_dmshifts, nchans, ndms, mstartdm, mdmstep, 2);
        }
        else if (choice.variant == -2) choice = choose_lds(h_dmshifts, nchans, ndms, mstartdm, mdmstep, -1);
        if (choice.variant >= 0) {
            rl->variant = choice.variant;
            rl->row_quads = choice.row_quads;
            return AA_HIP_SUCCESS;
        }
    }
    if (kernel == AA_HIP_KERNEL_LDS || forced >= 0)
        return fail(AA_HIP_ERROR_UNSUPPORTED, "the LDS kernel does not fit this geometry (delay spread per tile "
                                              "or row alignment)");
    return AA_HIP_SUCCESS;
}

lds_params lds_params_of(const range_launch &rl) {
    lds_params p{};
    p.L = rl.L;
    p.pitch = rl.pitch;
    p.nchans = rl.nchans;
    p.dmshifts = rl.d_dmshifts;
    p.ndms = rl.ndms;
    p.t_processed = rl.t_processed;
    p.mstartdm = rl.mstartdm;
    p.mdmstep = rl.mdmstep;
    p.fnchans = (float)rl.nchans;
    p.fbin = (float)rl.inBin;
    const auto pow2 = [](long v) { return v > 0 && (v & (v - 1)) == 0; };
    p.fscale = pow2(rl.nchans) && pow2(rl.inBin) ? (float)(1.0 / ((double)rl.nchans * (double)rl.inBin)) : 0.0f;
    p.out = rl.out;
    p.out_pitch = rl.out_pitch;
    p.row_quads = rl.row_quads;
    p.pair_recs = rl.pair_recs;
    if (rl.variant >= 0 && rl.variant < kLdsVariants) lds_job_tiles(p, rl.variant);
    return p;
}

hipError_t launch_range(const range_launch &rl, hipStream_t s) {
    if (rl.sample_bytes == 2) {
        const uint16_t *L = reinterpret_cast<const uint16_t *>(rl.L);
        if (rl.variant == kShapeMatrix) {
            lds_params p = lds_params_of(rl);
            p.L = rl.planes;
            p.pitch = rl.plane_pitch;
            const hipError_t e = launch_dedisperse_matrix(p, rl.mat, s, rl.over, rl.flags, rl.t_flags);
            if (e != hipSuccess) return e;
        }
        if (rl.wide_win > 0)
            return launch_dedisperse_wide_u16(L, rl.pitch / 2, rl.row_len, rl.nchans, rl.d_dmshifts, rl.ndms,
                                              rl.t_processed, rl.mstartdm, rl.mdmstep, rl.inBin, rl.out, rl.out_pitch,
                                              rl.wide_win, s, rl.flags, rl.mat.tile_out);
        return launch_dedisperse_direct_u16(L, rl.pitch / 2, rl.nchans, rl.d_dmshifts, rl.ndms, rl.t_processed,
                                            rl.mstartdm, rl.mdmstep, rl.inBin, rl.out, rl.out_pitch, s);
    }
    if (rl.variant == kShapeMatrix) return launch_dedisperse_matrix(lds_params_of(rl), rl.mat, s);
    if (rl.variant == kShapeRows) return launch_dedisperse_rows(lds_params_of(rl), s);
    if (rl.variant >= 0) return launch_dedisperse_lds(lds_params_of(rl), rl.variant, s);
    return launch_dedisperse_direct_u8(rl.L, rl.pitch, rl.nchans, rl.d_dmshifts, rl.ndms, rl.t_processed,
                                       rl.mstartdm, rl.mdmstep, rl.inBin, rl.out, rl.out_pitch, s);
}

int ddtr_engine::create(int device, int nchans, const float *dmshifts, int nranges,
                        const float *dm_low, const float *dm_step, const int *ndms,
                        const int *inBin, double tsamp, int maxshift, int max_t_processed0,
                        ddtr_engine **out, int sample_bits) {
    if (!out) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "out is NULL");
    *out = nullptr;
    if (sample_bits != 8 && sample_bits != 16) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "sample_bits must be 8 or 16");
    if (nchans <= 0 || nranges <= 0 || !dmshifts || !dm_low || !dm_step || !ndms || !inBin ||
        maxshift < 0 || max_t_processed0 <= 0 || !(tsamp > 0.0))
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "invalid plan geometry");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) {
        (void)hipGetLastError();
        return fail(AA_HIP_ERROR_NO_DEVICE, "no HIP device");
    }
    if (device < 0 || device >= count) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad device id");

    int max_bin = 1;
    for (int r = 0; r < nranges; ++r) {
        if (!is_pow2(inBin[r]))
            return fail(AA_HIP_ERROR_UNSUPPORTED, "inBin must be a power of two (range " + std::to_string(r) + ")");
        if (ndms[r] < 0) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "negative ndms");
        max_bin = std::max(max_bin, inBin[r]);
    }
    for (int c = 0; c < nchans; ++c)
        if (!(dmshifts[c] >= 0.0f) || !std::isfinite(dmshifts[c]))
            return fail(AA_HIP_ERROR_UNSUPPORTED,
                        "dmshift table must be finite and non-negative (descending channel frequencies)");

    device_guard guard(device);
    ddtr_engine *e = new ddtr_engine();
    e->m_device = device;
    e->m_sample_bytes = sample_bits / 8;
    e->m_nchans = nchans;
    e->m_tsamp = (float)tsamp;
    e->m_maxshift = maxshift;
    e->m_dmshifts.assign(dmshifts, dmshifts + nchans);
    for (int r = 0; r < nranges; ++r) e->m_ranges.push_back(range_desc{dm_low[r], dm_step[r], ndms[r], inBin[r]});

    hipError_t st = hipMalloc(&e->m_d_dmshifts, sizeof(float) * (size_t)nchans);
    if (st == hipSuccess) st = hipMemcpy(e->m_d_dmshifts, dmshifts, sizeof(float) * (size_t)nchans, hipMemcpyHostToDevice);
    if (st == hipSuccess) st = hipMalloc(&e->m_d_err, sizeof(int));
    if (st == hipSuccess) st = hipMemset(e->m_d_err, 0, sizeof(int));
    e->m_device_bytes = sizeof(float) * (size_t)nchans + sizeof(int);

    const int nlevels = log2i(max_bin) + 1;
    long cap = (long)max_t_processed0 + maxshift;
    for (int k = 0; k < nlevels && st == hipSuccess; ++k) {
        level lv;
        lv.capacity = cap;
        lv.pitch = round_up(((size_t)cap + kRowPad) * (size_t)e->m_sample_bytes, kPitchAlign);
        const size_t bytes = lv.pitch * (size_t)nchans;
        st = hipMalloc(&lv.ptr, bytes);
        if (st == hipSuccess) st = hipMemset(lv.ptr, 0, bytes);
        e->m_device_bytes += bytes;
        e->m_levels.push_back(lv);
        cap /= 2;
    }
    if (st == hipSuccess) st = hipDeviceSynchronize();
    if (st != hipSuccess) {
        const int code = hip_fail(st, "ddtr_engine allocation");
        delete e;
        return code;
    }
    *out = e;
    return AA_HIP_SUCCESS;
}

ddtr_engine::~ddtr_engine() {
    device_guard guard(m_device);
    for (auto &lv : m_levels) {
        if (lv.ptr) (void)hipFree(lv.ptr);
        if (lv.planes) (void)hipFree(lv.planes);
        if (lv.over) (void)hipFree(lv.over);
    }
    if (m_d_dmshifts) (void)hipFree(m_d_dmshifts);
    if (m_d_err) (void)hipFree(m_d_err);
    for (const auto &range : m_tables)
        for (const plan_tables &t : range)
            if (t.ptr) (void)hipFree(t.ptr);
    for (const matrix_tables &t : m_matrix) {
        if (t.t.ptr) (void)hipFree(t.t.ptr);
        if (t.flags) (void)hipFree(t.flags);
    }
}

int ddtr_engine::set_kernel(int kernel) {
    if (kernel < AA_HIP_KERNEL_AUTO || kernel > AA_HIP_KERNEL_MATRIX)
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "unknown kernel variant");
    m_kernel = kernel;
    return AA_HIP_SUCCESS;
}

void ddtr_engine::range_scalars(int r, float *mstartdm, float *mdmstep) const {
    const range_desc &rd = m_ranges[(size_t)r];
    const float tsamp_r = m_tsamp * (float)rd.inBin;
    *mstartdm = rd.dm_low / tsamp_r;
    *mdmstep = rd.dm_step / tsamp_r;
}

int ddtr_engine::ingest(const void *d_input_tc, int input_bits, int t_processed0, hipStream_t s) {
    if (!d_input_tc) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "input is NULL");
    const long len0 = (long)t_processed0 + m_maxshift;
    if (t_processed0 <= 0 || len0 > m_levels[0].capacity)
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "t_processed0 exceeds the handle's capacity");
    if (input_bits != 8 && input_bits != 16) return fail(AA_HIP_ERROR_UNSUPPORTED, "input_bits must be 8 or 16");
    device_guard guard(m_device);
    if (m_sample_bytes == 2) {   // u16 levels: samples keep their width
        if (input_bits != 16) return fail(AA_HIP_ERROR_UNSUPPORTED, "a 16-bit plan takes 16-bit input");
        const hipError_t e = launch_transpose_u16_pitch((const uint16_t *)d_input_tc, len0, m_nchans,
                                                        (uint16_t *)m_levels[0].ptr, m_levels[0].pitch / 2, s);
        if (e != hipSuccess) return hip_fail(e, "corner turn");
        for (auto &lv : m_levels) {
            lv.len = 0;
            lv.planes_ok = false;
        }
        m_levels[0].len = len0;
        m_resident = 0;
        return level_planes(0, s);
    }
    // The corner turn writes the binned levels the plan needs in the same
    // pass when the shapes allow it; otherwise ensure_level bins on demand.
    const int nlev = std::min((int)m_levels.size() - 1, kCtMaxLevels);
    uint8_t *ptrs[kCtMaxLevels + 1];
    size_t pitches[kCtMaxLevels + 1];
    for (int k = 0; k <= nlev; ++k) {
        ptrs[k] = m_levels[(size_t)k].ptr;
        pitches[k] = m_levels[(size_t)k].pitch;
    }
    int fused = 0;
    const hipError_t e = launch_corner_turn_levels(d_input_tc, input_bits / 8, len0, m_nchans, ptrs, pitches, nlev,
                                                   m_d_err, s, &fused, true);
    if (e != hipSuccess) return hip_fail(e, "corner turn");
    for (auto &lv : m_levels) lv.len = 0;
    for (int k = 0; k <= fused; ++k) m_levels[(size_t)k].len = len0 >> k;
    m_resident = fused;
    return AA_HIP_SUCCESS;
}

int ddtr_engine::ingest_job(const void *d_input_tc, int t_processed0, ct_job *job, bool *deferred) {
    *deferred = false;
    if (!d_input_tc) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "input is NULL");
    const long len0 = (long)t_processed0 + m_maxshift;
    if (t_processed0 <= 0 || len0 > m_levels[0].capacity)
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "t_processed0 exceeds the handle's capacity");
    if (m_sample_bytes != 1 || len0 > 0x7fffffffL) return AA_HIP_SUCCESS;   // ingest() handles these
    const int nlev = std::min((int)m_levels.size() - 1, kCtMaxLevels);
    ct_job j{};
    for (int k = 0; k <= nlev; ++k) {
        j.ptr[k] = m_levels[(size_t)k].ptr;
        j.pitch[k] = m_levels[(size_t)k].pitch;
        if ((size_t)(len0 >> k) > j.pitch[k]) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "level row too short");
    }
    if (!corner_turn_levels_wide(d_input_tc, m_nchans, j.ptr, j.pitch, nlev)) return AA_HIP_SUCCESS;
    j.in = static_cast<const uint8_t *>(d_input_tc);
    j.nsamp = len0;
    j.nchans = m_nchans;
    j.nlev = nlev;
    *job = j;
    for (auto &lv : m_levels) lv.len = 0;
    for (int k = 0; k <= nlev; ++k) m_levels[(size_t)k].len = len0 >> k;
    m_resident = nlev;
    *deferred = true;
    return AA_HIP_SUCCESS;
}

int ddtr_engine::take_input_overflow(hipStream_t s) {
    if (m_sample_bytes == 2) return 0;   // u16 levels hold any 16-bit value
    device_guard guard(m_device);
    int flag = 0;
    hipError_t e = hipMemcpyAsync(&flag, m_d_err, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e == hipSuccess && flag) e = hipMemsetAsync(m_d_err, 0, sizeof(int), s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e, "input flag");
    return flag ? 1 : 0;
}

int ddtr_engine::ensure_level(int k, hipStream_t s) {
    if (m_resident < 0) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "no chunk ingested");
    while (m_resident < k) {
        const level &src = m_levels[(size_t)m_resident];
        level &dst = m_levels[(size_t)m_resident + 1];
        const long n_out = src.len / 2;
        if (n_out > dst.capacity) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "binning level overflow");
        hipError_t e = m_sample_bytes == 2
                           ? launch_bin2_u16((const uint16_t *)src.ptr, src.pitch / 2, m_nchans, n_out,
                                             (uint16_t *)dst.ptr, dst.pitch / 2, s, true)
                           : launch_bin2_u8(src.ptr, src.pitch, m_nchans, (int)n_out, dst.ptr, dst.pitch, s);
        if (e != hipSuccess) return hip_fail(e, "binning");
        dst.len = n_out;
        ++m_resident;
        if (m_sample_bytes == 2) {
            const int st = level_planes(m_resident, s);
            if (st != AA_HIP_SUCCESS) return st;
        }
    }
    return AA_HIP_SUCCESS;
}

int ddtr_engine::prepare_range(int r, int t_processed, float *d_out, size_t out_pitch, hipStream_t s,
                               range_launch *rl, bool batched) {
    const int st = choose_launch(r, t_processed, d_out, out_pitch, s, rl, batched);
    if (st == AA_HIP_SUCCESS) {
        if (m_ran.size() != m_ranges.size()) m_ran.assign(m_ranges.size(), AA_HIP_RANGE_NONE);
        m_ran[(size_t)r] = rl->sample_bytes == 1 || rl->variant == kShapeMatrix ? rl->variant
                           : rl->wide_win > 0                                   ? (int)AA_HIP_RANGE_U16
                                                                                : (int)AA_HIP_RANGE_DIRECT;
    }
    return st;
}

int ddtr_engine::range_kernel(int r) const {
    static_assert(kShapeMatrix == AA_HIP_RANGE_MATRIX && kShapeRows == AA_HIP_RANGE_ROWS, "numbers of the kernels");
    return r >= 0 && r < (int)m_ran.size() ? m_ran[(size_t)r] : (int)AA_HIP_RANGE_NONE;
}

int ddtr_engine::choose_launch(int r, int t_processed, float *d_out, size_t out_pitch, hipStream_t s,
                               range_launch *rl, bool batched) {
    if (r < 0 || r >= (int)m_ranges.size()) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad range index");
    if (!d_out || out_pitch < (size_t)std::max(t_processed, 0))
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad output buffer");
    const range_desc &rd = m_ranges[(size_t)r];
    const int k = log2i(rd.inBin);
    device_guard guard(m_device);
    int st = ensure_level(k, s);
    if (st != AA_HIP_SUCCESS) return st;
    const level &lv = m_levels[(size_t)k];
    // Row length the reference gives this range: t_processed + maxshift/inBin.
    const long i_nsamp = (long)t_processed + m_maxshift / rd.inBin;
    if (i_nsamp > lv.len)
        return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "range " + std::to_string(r) + " needs " +
                                                       std::to_string(i_nsamp) + " samples per row, level holds " +
                                                       std::to_string(lv.len));
    float mstartdm, mdmstep;
    range_scalars(r, &mstartdm, &mdmstep);
    st = check_delays(m_dmshifts.data(), m_nchans, rd.ndms, mstartdm, mdmstep, t_processed, i_nsamp);
    if (st != AA_HIP_SUCCESS) return st;
    if (m_sample_bytes == 2) {   // u16 levels: dedisperse_u16, or the direct kernel when its window is too wide
        *rl = range_launch{};
        rl->L = lv.ptr;
        rl->pitch = lv.pitch;
        rl->nchans = m_nchans;
        rl->d_dmshifts = m_d_dmshifts;
        rl->ndms = rd.ndms;
        rl->t_processed = t_processed;
        rl->mstartdm = mstartdm;
        rl->mdmstep = mdmstep;
        rl->inBin = rd.inBin;
        rl->out = d_out;
        rl->out_pitch = out_pitch;
        rl->sample_bytes = 2;
        rl->row_len = i_nsamp;
        rl->wide_win = m_kernel == AA_HIP_KERNEL_DIRECT ? -1 : u16_window(r);
        if (rl->wide_win < 0 && m_kernel != AA_HIP_KERNEL_AUTO && m_kernel != AA_HIP_KERNEL_DIRECT)
            return fail(AA_HIP_ERROR_UNSUPPORTED, "the 16-bit LDS kernel does not fit this range's delay spread");
        if (rd.ndms <= 0) return AA_HIP_SUCCESS;
        const bool forced = m_kernel == AA_HIP_KERNEL_MATRIX;
        if (!u16_matrix(r, s)) return forced ? no_matrix() : AA_HIP_SUCCESS;
        st = ensure_planes(k, s);   // (the kernel setting may have changed since the level was written)
        if (st == AA_HIP_ERROR_OUT_OF_MEMORY) return forced ? no_matrix() : AA_HIP_SUCCESS;
        if (st != AA_HIP_SUCCESS) return st;
        const matrix_tables &mt = m_matrix[(size_t)r];
        rl->variant = kShapeMatrix;
        rl->pair_recs = mt.t.ptr;
        rl->mat = mt.lay;
        rl->planes = lv.planes;
        rl->plane_pitch = lv.plane_pitch;
        rl->over = lv.over;
        rl->flags = mt.flags;
        rl->t_flags = (int)std::min(lv.len - m_maxshift / rd.inBin, 0x7fffffffL);
        return AA_HIP_SUCCESS;
    }
    if (m_lds.size() != m_ranges.size()) m_lds.assign(m_ranges.size(), lds_choice{-2, 0});
    lds_choice &c = m_lds[(size_t)r];
    // A range that is small, or whose trials are far apart, goes straight from
    // the rows (in a batch the beams' ranges fill the chip together).
    const range_tuning tuned = tuning(r);
    const bool automatic = tuned.automatic && m_kernel == AA_HIP_KERNEL_AUTO && rd.ndms > 0;
    const bool alone = automatic && !batched;
    const auto shape = [&]() {   // the range's LDS shape: c, chosen on first use
        if (c.variant == -2) {
            c = choose_lds(m_dmshifts.data(), m_nchans, rd.ndms, mstartdm, mdmstep, tuned.variant);
            if (c.variant < 0 && tuned.variant >= 0)  // preferred shape does not fit: any that does
                c = choose_lds(m_dmshifts.data(), m_nchans, rd.ndms, mstartdm, mdmstep, -1);
        }
        return c.variant;
    };
    // No shape asked for: the matrix kernel where its plan is the cheaper one.
    const bool forced = m_kernel == AA_HIP_KERNEL_MATRIX && rd.ndms > 0;
    if (forced || (automatic && (!batched || matrix_tiles_at_most(rd.ndms, t_processed) >= kMatrixAloneTiles))) {
        const hipError_t e = plan_matrix(r, lv.pitch, 1, s);
        if (e != hipSuccess && (forced || e != hipErrorOutOfMemory)) return hip_fail(e, "plan tables");
        const matrix_tables &mt = m_matrix[(size_t)r];
        if (forced && mt.lay.tile_out <= 0) return no_matrix();
        const long tiles =
            mt.lay.tile_out > 0 ? (long)mt.lay.n_dm_tiles * ((t_processed + mt.lay.tile_out - 1) / mt.lay.tile_out) : 0;
        const bool takes =
            forced || (tiles > 0 && (batched ? tiles >= kMatrixAloneTiles &&
                                                   matrix_beats_shared(m_nchans, rd.ndms, t_processed, mt.lay, shape())
                                             : !rows_beat_matrix(m_nchans, rd.ndms, t_processed, mt.lay)));
        if (takes) {
            st = resolve_launch(m_kernel, lv.ptr, lv.pitch, m_nchans, m_d_dmshifts, m_dmshifts.data(), rd.ndms,
                                t_processed, mstartdm, mdmstep, rd.inBin, d_out, out_pitch,
                                lds_choice{kShapeMatrix, mt.lay.tile_out}, rl);
            rl->pair_recs = mt.t.ptr;
            rl->mat = mt.lay;
            return st;
        }
    }
    shape();
    // Under capture a shape whose tables are not there yet (the calls before went
    // another way) would break the capture; the rows need none.
    const bool rows = ((alone || (automatic && c.variant < 0)) &&
                       rows_beat_shape(m_nchans, rd.ndms, t_processed, c.variant)) ||
                      (automatic && c.variant >= 2 && !has_tables(r, c.variant) && capturing(s));
    st = resolve_launch(m_kernel, lv.ptr, lv.pitch, m_nchans, m_d_dmshifts, m_dmshifts.data(), rd.ndms,
                        t_processed, mstartdm, mdmstep, rd.inBin, d_out, out_pitch,
                        rows ? lds_choice{kShapeRows, 0} : c, rl);
    if (st != AA_HIP_SUCCESS || rl->variant < 2 || rl->variant == kShapeRows) return st;
    // Chunk shapes from 2 on read plan tables; they depend on the range and
    // shape only, so they are built once, on the first call that needs them.
    if (m_tables.size() != m_ranges.size()) m_tables.resize(m_ranges.size());
    plan_tables &pt = m_tables[(size_t)r][(size_t)rl->variant];
    if (!pt.ptr) {
        std::vector<uint8_t> bytes;
        if (lds_plan_tables(rl->variant, m_dmshifts.data(), m_nchans, rd.ndms, mstartdm, mdmstep, lv.pitch, &bytes) !=
            rl->row_quads)
            return fail(AA_HIP_ERROR_UNSUPPORTED, "plan tables disagree with the chosen row width");
        const hipError_t e = keep_tables(pt, bytes);
        if (e != hipSuccess) return hip_fail(e, "plan tables");
    }
    rl->pair_recs = pt.ptr;
    return AA_HIP_SUCCESS;
}

bool ddtr_engine::has_tables(int r, int variant) const {
    return !m_tables.empty() && m_tables[(size_t)r][(size_t)variant].ptr;
}

// The window of dedisperse_u16 for range r of a u16 plan (-1: direct kernel).
int ddtr_engine::u16_window(int r) {
    if (m_wide_win.size() != m_ranges.size()) m_wide_win.assign(m_ranges.size(), 0);
    int &w = m_wide_win[(size_t)r];
    if (w == 0) {
        float mstartdm, mdmstep;
        range_scalars(r, &mstartdm, &mdmstep);
        w = wide_window(m_dmshifts.data(), m_nchans, m_ranges[(size_t)r].ndms, mstartdm, mdmstep);
    }
    return w;
}

// The automatic choice on u16 levels: the matrix kernel over the rows' byte
// planes where its plan pays (dedisperse_u16 then computes the tiles it
// flags).  Without the memory for its tables or the level's planes the range
// keeps dedisperse_u16, from its first chunk on; captured before they are there,
// a call takes dedisperse_u16 this time.
bool ddtr_engine::u16_matrix(int r, hipStream_t s) {
    if (m_sample_bytes != 2 || (m_kernel != AA_HIP_KERNEL_AUTO && m_kernel != AA_HIP_KERNEL_MATRIX) ||
        u16_window(r) <= 0)
        return false;
    const bool forced = m_kernel == AA_HIP_KERNEL_MATRIX;
    if (!forced && m_nchans < kU16MatrixMinChannels) return false;
    const range_desc &rd = m_ranges[(size_t)r];
    const level &lv = m_levels[(size_t)log2i(rd.inBin)];
    (void)plan_matrix(r, round_up((size_t)lv.capacity + kRowPad, kPitchAlign), 2, s);
    matrix_tables &mt = m_matrix[(size_t)r];
    // The chunk's length decides, not the call's: its planes are made at ingest.
    if (mt.lay.tile_out <= 0 || !(forced || matrix_beats_u16(m_nchans, lv.len - m_maxshift / rd.inBin, mt.lay)))
        return false;
    if (mt.flags) return true;
    const size_t tiles =
        (size_t)mt.lay.n_dm_tiles * (size_t)((lv.capacity + mt.lay.tile_out - 1) / mt.lay.tile_out) * sizeof(int);
    if (hipMalloc(&mt.flags, tiles) != hipSuccess) {
        (void)hipGetLastError();
        mt.flags = nullptr;
        drop_matrix(r);
        return false;
    }
    mt.flag_bytes = tiles;
    m_device_bytes += tiles;
    return true;
}

// Byte planes of a u16 level that has just been written, where a range reads
// them: on the writer's stream, so that ranges may run on others.
int ddtr_engine::level_planes(int k, hipStream_t s) {
    m_levels[(size_t)k].planes_ok = false;
    for (int r = 0; r < (int)m_ranges.size(); ++r)
        if (log2i(m_ranges[(size_t)r].inBin) == k && m_ranges[(size_t)r].ndms > 0 && u16_matrix(r, s)) {
            const int st = ensure_planes(k, s);
            return st == AA_HIP_ERROR_OUT_OF_MEMORY ? AA_HIP_SUCCESS : st;
        }
    return AA_HIP_SUCCESS;
}

// Byte planes of level k for the current chunk.  Without the memory for them
// no range of the level takes the matrix kernel (captured before they are there,
// this time): OUT_OF_MEMORY, no message set.

int ddtr_engine::ensure_planes(int k, hipStream_t s) {
    level &lv = m_levels[(size_t)k];
    if (lv.planes_ok) return AA_HIP_SUCCESS;
    if (!lv.planes) {
        if (capturing(s)) return AA_HIP_ERROR_OUT_OF_MEMORY;
        const size_t pitch = round_up((size_t)lv.capacity + kRowPad, kPitchAlign);
        void *p = nullptr, *o = nullptr;
        if (hipMalloc(&p, 2 * pitch * (size_t)m_nchans) != hipSuccess || hipMalloc(&o, 64 * sizeof(int)) != hipSuccess) {
            (void)hipGetLastError();
            if (p) (void)hipFree(p);
            for (int r = 0; r < (int)m_matrix.size(); ++r)
                if (log2i(m_ranges[(size_t)r].inBin) == k) drop_matrix(r);
            return AA_HIP_ERROR_OUT_OF_MEMORY;
        }
        lv.planes = static_cast<uint8_t *>(p);
        lv.over = static_cast<int *>(o);
        lv.plane_pitch = pitch;
        m_device_bytes += 2 * pitch * (size_t)m_nchans + 64 * sizeof(int);
    }
    const uint16_t *rows = reinterpret_cast<const uint16_t *>(lv.ptr);
    hipError_t e = launch_u16_sums_over(rows, lv.pitch / 2, m_nchans, lv.len, lv.over, s);
    if (e == hipSuccess)
        e = launch_split_u16(rows, lv.pitch / 2, m_nchans, lv.len, lv.planes,
                             lv.planes + lv.plane_pitch * (size_t)m_nchans, lv.plane_pitch, lv.over, s);
    if (e != hipSuccess) return hip_fail(e, "byte planes");
    lv.planes_ok = true;
    return AA_HIP_SUCCESS;
}

hipError_t ddtr_engine::keep_tables(plan_tables &pt, const std::vector<uint8_t> &bytes) {
    void *t = nullptr;
    hipError_t e = hipMalloc(&t, bytes.size());
    if (e == hipSuccess) e = hipMemcpy(t, bytes.data(), bytes.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // else the next launch reports it
        if (t) (void)hipFree(t);
        return e;
    }
    pt.ptr = t;
    pt.bytes = bytes.size();
    m_device_bytes += bytes.size();
    return hipSuccess;
}

void ddtr_engine::drop_tables(plan_tables &pt) {
    if (pt.ptr) (void)hipFree(pt.ptr);
    m_device_bytes -= pt.bytes;
    pt = plan_tables{};
}

// Range r's plan for the matrix kernel, made once, with its tables on the
// device; tile_out 0 where the plan does not pay.  Without the memory for it
// (host or device) the range is not the matrix kernel's either, from its first
// call on: hipErrorOutOfMemory, once, for callers that have no other kernel.
// Under capture nothing is planned; the next eager call does.
hipError_t ddtr_engine::plan_matrix(int r, size_t pitch, int planes, hipStream_t s) {
    if (m_matrix.size() != m_ranges.size()) m_matrix.resize(m_ranges.size());
    matrix_tables &mt = m_matrix[(size_t)r];
    if (mt.planned || capturing(s)) return hipSuccess;
    mt.planned = true;
    float mstartdm, mdmstep;
    range_scalars(r, &mstartdm, &mdmstep);
    try {
        std::vector<uint8_t> bytes;
        const matrix_layout lay =
            matrix_plan(m_dmshifts.data(), m_nchans, m_ranges[(size_t)r].ndms, mstartdm, mdmstep, pitch, &bytes, planes);
        const hipError_t e = lay.tile_out > 0 ? keep_tables(mt.t, bytes) : hipSuccess;
        if (e == hipSuccess) mt.lay = lay;
        return e;
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
}

// Range r is not the matrix kernel's after all; gives back what it held for it.
void ddtr_engine::drop_matrix(int r) {
    matrix_tables &mt = m_matrix[(size_t)r];
    drop_tables(mt.t);
    if (mt.flags) (void)hipFree(mt.flags);
    m_device_bytes -= mt.flag_bytes;
    mt = matrix_tables{};
    mt.planned = true;
}

int ddtr_engine::set_range_tuning(int r, int variant, bool automatic) {
    if (r < 0 || r >= (int)m_ranges.size()) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad range index");
    if (variant < -1 || variant >= kLdsVariants) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad LDS variant");
    if (m_tuning.size() != m_ranges.size()) m_tuning.assign(m_ranges.size(), range_tuning{});
    m_tuning[(size_t)r] = range_tuning{variant, automatic || variant < 0};
    if (m_lds.size() == m_ranges.size()) m_lds[(size_t)r] = lds_choice{-2, 0};
    return AA_HIP_SUCCESS;
}

range_tuning ddtr_engine::tuning(int r) const {
    return r >= 0 && r < (int)m_tuning.size() ? m_tuning[(size_t)r] : range_tuning{};
}

int ddtr_engine::autotune_range(int r, int t_processed, float *d_out, size_t out_pitch, int reps, hipStream_t s,
                                int *best, float *ms) {
    if (!best || !ms || reps <= 0) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad autotune arguments");
    if (m_sample_bytes == 2) return fail(AA_HIP_ERROR_UNSUPPORTED, "16-bit plans have one kernel (nothing to tune)");
    if (r < 0 || r >= (int)m_ranges.size()) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "bad range index");
    device_guard guard(m_device);
    const int saved_kernel = m_kernel;
    m_kernel = AA_HIP_KERNEL_AUTO;
    *best = -1;
    bool had[kLdsVariants];
    for (int v = 0; v < kLdsVariants; ++v) had[v] = has_tables(r, v);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    int st = AA_HIP_SUCCESS;
    float best_ms = 0.0f;
    float auto_ms = -1.0f;   // the automatic choice where that is none of the shapes
    for (int v = -1; v < kLdsVariants && e == hipSuccess && st == AA_HIP_SUCCESS; ++v) {
        if (v >= 0) ms[v] = -1.0f;
        st = set_range_tuning(r, v, false);
        range_launch rl;
        if (st == AA_HIP_SUCCESS) st = prepare_range(r, t_processed, d_out, out_pitch, s, &rl);
        if (st != AA_HIP_SUCCESS || (v < 0 ? rl.variant < kLdsVariants : rl.variant != v)) continue;
        e = launch_range(rl, s);
        if (e == hipSuccess) e = hipEventRecord(e0, s);
        for (int i = 0; i < reps && e == hipSuccess; ++i) e = launch_range(rl, s);
        if (e == hipSuccess) e = hipEventRecord(e1, s);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        float t = 0.0f;
        if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
        if (e != hipSuccess) break;
        (v < 0 ? auto_ms : ms[v]) = t / (float)reps;
        if (v >= 0 && (*best < 0 || ms[v] < best_ms)) {
            *best = v;
            best_ms = ms[v];
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    m_kernel = saved_kernel;
    if (st == AA_HIP_SUCCESS && e != hipSuccess) st = hip_fail(e, "autotune");
    for (int v = 0; !m_tables.empty() && v < kLdsVariants; ++v)   // tables made for this, in no graph
        if (v != *best && !had[v]) drop_tables(m_tables[(size_t)r][(size_t)v]);
    // The best shape is kept beside the automatic choice too: a batch leaves the
    // matrix and row kernels out where its ranges share launches.
    if (st == AA_HIP_SUCCESS) st = set_range_tuning(r, *best, auto_ms >= 0.0f && (*best < 0 || auto_ms <= best_ms));
    return st;
}

int ddtr_engine::run_range(int r, int t_processed, float *d_out, size_t out_pitch, hipStream_t s) {
    range_launch rl;
    const int st = prepare_range(r, t_processed, d_out, out_pitch, s, &rl);
    if (st != AA_HIP_SUCCESS) return st;
    device_guard guard(m_device);
    const hipError_t e = launch_range(rl, s);
    if (e != hipSuccess) return hip_fail(e, "dedisperse");
    return AA_HIP_SUCCESS;
}

int ddtr_engine::execute_chunk(const void *d_input_tc, int input_bits, const int *t_processed,
                               float *const *d_out, const size_t *out_pitch, hipStream_t s) {
    if (!t_processed || !d_out || !out_pitch) return fail(AA_HIP_ERROR_INVALID_ARGUMENT, "NULL array");
    int st = ingest(d_input_tc, input_bits, t_processed[0], s);
    for (int r = 0; r < (int)m_ranges.size() && st == AA_HIP_SUCCESS; ++r)
        st = run_range(r, t_processed[r], d_out[r], out_pitch[r], s);
    return st;
}

}  // namespace aa_hip

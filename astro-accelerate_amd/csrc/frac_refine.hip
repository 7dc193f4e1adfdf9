// Batched DM refinement of candidate windows of uneven size, for gfx950.
// No counterpart in the reference.  Each candidate b is a float32 window
// x_b[c][t] (C_b channels x T_b samples) cut along the candidate's
// dispersion track; its continuous residual DM u_b is refined by gradient
// ascent on the energy of the dedispersed profile,
//     E(u) = sum_t y(t)^2,  y(t) = sum_c (1 - f_c) x[c][t + i_c] + f_c x[c][t + i_c + 1],
//     tau_c = ds[c] * u (double), i_c = floor(tau_c), f_c = tau_c - i_c,
// with x = 0 outside [0, T) and ds[c] the delay per unit DM in samples.
//     dE/du = sum_c ds[c] sum_t 2 y(t) (x[c][t + i_c + 1] - x[c][t + i_c]).
//
// Two losses (refine_args::loss_kind):
//  0  L = E.
//  1  L = E - N, the energy in excess of what white noise of the window's
//     channel powers v_c = mean_t x[c][t]^2 would give at the same delays:
//         N(u) = sum_c v_c ((1 - f_c)^2 (T - |i_c|)+ + f_c^2 (T - |i_c + 1|)+),
//     the expected sum_t y(t)^2 of independent channels of variances v_c
//     (each channel's two taps cover (T - |i|)+ and (T - |i + 1|)+ output
//     samples).  Interpolation averages neighbouring noise samples, so E of
//     pure noise is largest where every f_c is 0 (u = 0) and about a third
//     lower in between: on weak candidates that spike outweighs the pulse.
//     dN/du = sum_c v_c ds[c] (2 f_c (T - |i_c + 1|)+ - 2 (1 - f_c) (T - |i_c|)+).
//     v_c is computed once per run (refine_power_kernel).
//
// An optional coarse scan first evaluates L (forward pass only) at scan_n
// offsets u + scan_lo + k * scan_step and starts the steps from the best.
//
// One evaluation is one pass over the windows: dy/du (t) = sum_c ds[c] (x[c][t +
// i_c + 1] - x[c][t + i_c]) does not depend on y, so the pass accumulates y and
// dy/du together and dE/du = 2 sum_t y dy/du follows from them.  The scan's
// points (kScan at a time) share one pass too.
//
// Work split: an item is up to kChunk channels (fewer where the windows are few,
// refine_chunk) x kSeg samples of one window, a 256-thread work-group each, so
// that windows of any number and size spread over the whole GPU.  A group of S
// lanes covers the item's samples, 4 consecutive ones per lane, and the work-group
// holds G = 256 / S such groups, each summing every G-th channel.  A lane reads its 4 samples x[c][t0 + i_c ..
// t0 + i_c + 3] as one 16-byte load; the second tap of the sample before them
// is kept apart and added to it after the pass.  Sums are double; the groups'
// are added in LDS and the items' by one work-group per candidate
// (refine_combine_kernel), which also applies the sign-based adaptive step
// (Rprop: the step grows by 1.2 while the sign of dL/du holds and halves when
// it flips); the result is the best point visited.  Every sum runs in a fixed
// order: results do not depend on scheduling.  An evaluation is two launches.
//
// Bound: HBM (each pass reads every window once; the partial profiles add 2 to
// 3 % of that).  Measured on 256 windows (1024-4096 channels x 256-4096
// samples, 3.64 GB; 9-point scan and 20 steps): 21.7 ms, of which a gradient
// pass takes 0.75 ms (4.85 TB/s; a 4 GiB device copy does 4.77), its combine
// 0.04, a scan pass of 3 points 1.45, the channel powers 1.05.  With one
// work-group per window, two passes per evaluation and one per scan point it
// took 178 ms (the largest windows' work-groups ran long after the others).
// Scan points per pass: 9 in one took 6.1 ms (150 registers), 5 and 4 took
// 2 x 2.4, 3 take 3 x 1.45; two channels in flight per lane in a scan pass 1.88
// instead of 1.45 (the window-edge branch of each load).
#include "frac_refine.h"

#include <cmath>

#include "linear_grid.h"

namespace aa_hip {

namespace {

constexpr int kThreads = kRefineThreads;
constexpr int kSpt = 4;                       // consecutive samples per lane
constexpr int kU = 4;                         // channels in flight per lane
constexpr int kSeg = kRefineSeg;
constexpr int kChunk = kRefineChunk;
constexpr int kScan = kRefineScan;
constexpr int kCombineThreads = 1024;         // threads of a window's combine pass; 256 for short windows,
constexpr int kCombineShort = 256;            // whose samples would leave most of them idle
static_assert(kSeg == kThreads * kSpt, "a segment's samples fit one lane span each");

// w[m] = row[j + m], m = 0..3, zero outside [0, T).
__device__ __forceinline__ void load4(const float* __restrict__ row, int j, int T, float (&w)[4])
{
    if (j >= 0 && j + 3 < T) {
        float4 q;
        __builtin_memcpy(&q, row + j, sizeof(q));   // dword-aligned 16-byte load
        w[0] = q.x;
        w[1] = q.y;
        w[2] = q.z;
        w[3] = q.w;
    } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int i = j + m;
            w[m] = (i >= 0 && i < T) ? row[i] : 0.0f;
        }
    }
}

__device__ __forceinline__ float load1(const float* __restrict__ row, int i, int T)
{
    return (i >= 0 && i < T) ? row[i] : 0.0f;
}

// Integer and fractional delay of a channel at residual DM u.
__device__ __forceinline__ int2 delay_of(float ds, float u)
{
    const double tau = (double)ds * (double)u;
    const double fl = fmin(fmax(floor(tau), -1073741824.0), 1073741824.0);
    return make_int2((int)fl, __float_as_int((float)(tau - fl)));
}

// Profile sample t of a window lies at t + t / kSeg of a partial profile; the
// entry after a full segment takes the next segment's share of its last sample.
// Sums of NP profiles `row` entries apart over the window's chunks, in order.
template <int NP>
__device__ __forceinline__ void profile_at(const double* __restrict__ part, size_t stride, int row, int nchunk, int t,
                                           int T, double (&v)[NP])
{
    const double* q = part + t + t / kSeg;
    double e[NP];
#pragma unroll
    for (int n = 0; n < NP; ++n) v[n] = e[n] = 0.0;
#pragma unroll 8
    for (int j = 0; j < nchunk; ++j)
#pragma unroll
        for (int n = 0; n < NP; ++n) v[n] += q[(size_t)j * stride + (size_t)n * row];
    if ((t + 1) % kSeg == 0 && t + 1 < T) {
        for (int j = 0; j < nchunk; ++j)
#pragma unroll
            for (int n = 0; n < NP; ++n) e[n] += q[(size_t)j * stride + (size_t)n * row + 1];
    }
#pragma unroll
    for (int n = 0; n < NP; ++n) v[n] += e[n];
}

// Partial profiles of one item.  NK = 0: y and dy/du at the candidate's current
// u (2 arrays); NK = kScan: y at scan points k0 .. k0 + nk - 1 (nk arrays).
template <int NK>
__global__ __launch_bounds__(kThreads) void refine_partial_kernel(refine_args a, int k0, int nk)
{
    constexpr int K = NK ? NK : 1;
    __shared__ int2 tab[K][kChunk];        // (i_c, f_c bits)
    __shared__ float dsv[kChunk];
    __shared__ double r_y[kSeg], r_p[NK ? 1 : kSeg + 8];
    __shared__ double r_b[2][kThreads / 64];
    const long item = linear_block();
    if (item >= a.nitems) return;   // whole work-group, before any barrier
    const refine_item it = a.items[item];
    const refine_cand cd = a.cands[it.cand];
    const int tid = threadIdx.x, T = cd.T, C = it.nc, t_first = it.seg * kSeg;
    const int nt = min(kSeg, T - t_first);
    const bool last_seg = t_first + nt == T;
    const float* __restrict__ x = a.x + cd.x_off + (size_t)it.c0 * T;
    const float u0 = NK ? a.u[it.cand] : a.cur[it.cand].u;
    for (int c = tid; c < C; c += kThreads) {
        const float d = a.ds[cd.ds_off + it.c0 + c];
        dsv[c] = d;
#pragma unroll
        for (int k = 0; k < K; ++k)
            tab[k][c] = delay_of(d, NK ? u0 + a.scan_lo + a.scan_step * (float)(k0 + k) : u0);
    }
    __syncthreads();

    // samples t_first .. t_first + nt - 1 and, in the window's last segment, T:
    // its taps are the second ones of sample T - 1.  A full last segment has no
    // lane for it: its last lane reads it in addition (edge).
    const int ns = min(kSeg, nt + (last_seg ? 1 : 0));
    const int S = ((ns + kSpt - 1) / kSpt + 63) / 64 * 64;
    const int G = kThreads / S, g = tid / S, s = tid - g * S;
    const bool active = g < G && kSpt * s < ns;
    const int t0 = t_first + kSpt * s;
    const bool any_edge = last_seg && nt == kSeg, edge = any_edge && s == S - 1;
    double y[K][kSpt], yn[K], P[kSpt], pe = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        yn[k] = 0.0;
#pragma unroll
        for (int m = 0; m < kSpt; ++m) y[k][m] = 0.0;
    }
#pragma unroll
    for (int m = 0; m < kSpt; ++m) P[m] = 0.0;
    auto add = [&](int k, int c, const float (&w)[4]) {
        const int2 e = tab[k][c];
        const double f = (double)__int_as_float(e.y);
#pragma unroll
        for (int m = 0; m < kSpt; ++m) y[k][m] = __builtin_fma(1.0 - f, (double)w[m], y[k][m]);
#pragma unroll
        for (int m = 1; m < kSpt; ++m) y[k][m - 1] = __builtin_fma(f, (double)w[m], y[k][m - 1]);
        yn[k] = __builtin_fma(f, (double)w[0], yn[k]);
        if (!NK) {
            const double d = (double)dsv[c];
#pragma unroll
            for (int m = 0; m < kSpt; ++m) P[m] = __builtin_fma(d, (double)w[m], P[m]);
        }
        if (any_edge && edge) {
            const double v = (double)load1(x + (size_t)c * T, T + e.x, T);
            y[k][kSpt - 1] = __builtin_fma(f, v, y[k][kSpt - 1]);
            if (!NK) pe = __builtin_fma((double)dsv[c], v, pe);
        }
    };
    if (active) {
        constexpr int U = NK ? 1 : kU;
        int c = g;
        for (; c + (U - 1) * G < C; c += U * G) {
            float w[U * K][4];
#pragma unroll
            for (int i = 0; i < U; ++i)
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (!NK || k < nk)
                        load4(x + (size_t)(c + i * G) * T, t0 + tab[k][c + i * G].x, T, w[i * K + k]);
#pragma unroll
            for (int i = 0; i < U; ++i)
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (!NK || k < nk) add(k, c + i * G, w[i * K + k]);
        }
        for (; c < C; c += G) {
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (!NK || k < nk) {
                    float w[4];
                    load4(x + (size_t)c * T, t0 + tab[k][c].x, T, w);
                    add(k, c, w);
                }
        }
    }

    const int row = T + (T - 1) / kSeg;              // entries of a profile
    const int S4 = kSpt * S;                         // one group's samples in LDS (G * S4 <= kSeg)
    double* __restrict__ out = a.part + cd.part_off + (size_t)it.chunk * (NK ? kScan : 2) * row;
    const int o = t_first + it.seg;                  // first entry of the segment
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (NK && k >= nk) continue;   // (not break: k stays a constant in the unrolled body)
        __syncthreads();
        if (g < G) {
#pragma unroll
            for (int m = 0; m < kSpt; ++m) r_y[g * S4 + kSpt * s + m] = y[k][m];
            if (!NK) {
#pragma unroll
                for (int m = 0; m < kSpt; ++m) r_p[g * S4 + kSpt * s + m] = P[m];
            }
        }
        __syncthreads();
        if (g < G) {
            if (s > 0) r_y[g * S4 + kSpt * s - 1] += yn[k];   // one lane per entry
            else r_b[0][g] = yn[k];
            if (!NK && s == 0) r_b[1][g] = P[0];
            if (!NK && G == 1 && s == S - 1) r_p[S4] = pe;    // sample T, or the next segment's
        }
        __syncthreads();
        for (int t = tid; t < nt; t += kThreads) {
            double v = 0.0, p = 0.0;
            for (int h = 0; h < G; ++h) {
                v += r_y[h * S4 + t];
                if (!NK) p += r_p[h * S4 + t + 1] - r_p[h * S4 + t];
            }
            out[(size_t)k * row + o + t] = v;
            if (!NK) out[(size_t)row + o + t] = p;
        }
        if (tid == 0 && it.seg > 0) {
            double v = 0.0, p = 0.0;
            for (int h = 0; h < G; ++h) {
                v += r_b[0][h];
                if (!NK) p += r_b[1][h];
            }
            out[(size_t)k * row + o - 1] = v;
            if (!NK) out[(size_t)row + o - 1] = p;
        }
    }
}

template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red, int tid)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __syncthreads();                        // red free (previous reduction read)
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < NT / 64; ++i) s += red[i];
    return s;
}

// This thread's channels of the noise energy N (loss 1) and dN/du at u.
template <int NT>
__device__ __forceinline__ void noise_part(const refine_args& a, const refine_cand& cd, float u, int tid, double* n,
                                           double* dn)
{
    *n = *dn = 0.0;
    if (a.loss_kind != 1) return;
    for (int c = tid; c < cd.C; c += NT) {
        const float ds = a.ds[cd.ds_off + c];
        const int2 e = delay_of(ds, u);
        const double f = (double)__int_as_float(e.y);       // the weight the passes use
        const double n0 = (double)max(0, cd.T - abs(e.x)), n1 = (double)max(0, cd.T - abs(e.x + 1));
        const double v = a.power[cd.power_off + c];
        *n = __builtin_fma(v, (1.0 - f) * (1.0 - f) * n0 + f * f * n1, *n);
        *dn = __builtin_fma(v * (double)ds, 2.0 * f * n1 - 2.0 * (1.0 - f) * n0, *dn);
    }
}

// Loss at scan point k0 + blockIdx.y of candidate blockIdx.x.
template <int NT>
__global__ __launch_bounds__(NT) void refine_scan_loss_kernel(refine_args a, int k0)
{
    __shared__ double red[NT / 64];
    const long b = linear_block();
    if (b >= a.ncand) return;   // whole work-group, before any barrier
    const int k = blockIdx.y, tid = threadIdx.x;
    const refine_cand cd = a.cands[b];
    const int row = cd.T + (cd.T - 1) / kSeg, nchunk = (cd.C + a.chunk - 1) / a.chunk;
    const double* part = a.part + cd.part_off + (size_t)k * row;
    double l2 = 0.0, n, dn;
    for (int t = tid; t < cd.T; t += NT) {
        double v[1];
        profile_at(part, (size_t)kScan * row, row, nchunk, t, cd.T, v);
        l2 = __builtin_fma(v[0], v[0], l2);
    }
    noise_part<NT>(a, cd, a.u[b] + a.scan_lo + a.scan_step * (float)(k0 + k), tid, &n, &dn);
    const double l = block_sum<NT>(l2 - n, red, tid);
    if (tid == 0) a.scan_loss[(size_t)b * kScan + k] = l;
}

// Starts the candidates' states (k0 = 0), then takes in the losses of scan
// points k0 .. k0 + nk - 1, in order.
__global__ void refine_start_kernel(refine_args a, int k0, int nk)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= a.ncand) return;
    refine_state st = k0 == 0 ? refine_state{a.u[b], a.step[b], a.u[b], a.prev_grad[b], -INFINITY, 0.0} : a.cur[b];
    for (int k = 0; k < nk; ++k) {
        const double l = a.scan_loss[(size_t)b * kScan + k];
        if (l > st.best_l) {
            st.best_l = l;
            st.best_u = a.u[b] + a.scan_lo + a.scan_step * (float)(k0 + k);
        }
    }
    if (k0 + nk >= a.scan_n) {   // the steps start from the best point
        st.u = st.best_u;
        st.best_l = -INFINITY;
    }
    a.cur[b] = st;
}

// One candidate's loss and gradient from the partial profiles, and its step.
template <int NT>
__global__ __launch_bounds__(NT) void refine_combine_kernel(refine_args a, int last)
{
    __shared__ double red[NT / 64];
    const long b = linear_block();
    if (b >= a.ncand) return;   // whole work-group, before any barrier
    const int tid = threadIdx.x;
    const refine_cand cd = a.cands[b];
    const int row = cd.T + (cd.T - 1) / kSeg, nchunk = (cd.C + a.chunk - 1) / a.chunk;
    const double* part = a.part + cd.part_off;
    refine_state st = a.cur[b];
    double l2 = 0.0, gs = 0.0, n, dn;
    for (int t = tid; t < cd.T; t += NT) {
        double v[2];   // y, dy/du
        profile_at(part, 2 * (size_t)row, row, nchunk, t, cd.T, v);
        l2 = __builtin_fma(v[0], v[0], l2);
        gs = __builtin_fma(v[0], v[1], gs);
    }
    noise_part<NT>(a, cd, st.u, tid, &n, &dn);
    const double loss = block_sum<NT>(l2 - n, red, tid);
    const double grad = block_sum<NT>(2.0 * gs - dn, red, tid);
    if (tid != 0) return;
    if (loss > st.best_l) {  // the result is the best point visited
        st.best_l = loss;
        st.best_u = st.u;
        a.best_grad[b] = grad;
    } else if (st.best_l == -INFINITY) {
        a.best_grad[b] = 0.0;
    }
    if (last) {
        a.u[b] = st.best_u;
        a.step[b] = st.step;
        a.prev_grad[b] = st.prev;
        a.loss[b] = st.best_l;
        a.grad[b] = a.best_grad[b];
        return;
    }
    if (grad * st.prev > 0.0) st.step = fminf(st.step * 1.2f, a.step_max);
    else if (grad * st.prev < 0.0) st.step = fmaxf(st.step * 0.5f, a.step_min);
    st.u = st.u + (grad > 0.0 ? st.step : (grad < 0.0 ? -st.step : 0.0f));
    st.prev = grad;
    a.cur[b] = st;
}

// v_c = mean_t x[c][t]^2 of every candidate's channels: work-group (b, y)
// of candidate b takes channels 4 y + wave + 64 k, one wave per channel at a
// time with four 256-byte loads in flight per lane; fixed reduction order.
constexpr int kPowerBlocksY = 16;
__global__ __launch_bounds__(256) void refine_power_kernel(refine_args a)
{
    const long b = linear_block();
    if (b >= a.ncand) return;
    const refine_cand cd = a.cands[b];
    const float* __restrict__ x = a.x + cd.x_off;
    double* __restrict__ v = a.power + cd.power_off;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int T = cd.T;
    for (int c = 4 * (int)blockIdx.y + wave; c < cd.C; c += 4 * kPowerBlocksY) {
        const float* row = x + (size_t)c * T;
        double s[4] = {0.0, 0.0, 0.0, 0.0};
        int t = lane;
        for (; t + 192 < T; t += 256) {
            float q[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) q[m] = row[t + 64 * m];
#pragma unroll
            for (int m = 0; m < 4; ++m) s[m] = __builtin_fma((double)q[m], (double)q[m], s[m]);
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) {   // fewer than 256 samples left
            if (t + 64 * m < T) {
                const double q = (double)row[t + 64 * m];
                s[m] = __builtin_fma(q, q, s[m]);
            }
        }
        double r = (s[0] + s[1]) + (s[2] + s[3]);
        for (int off = 32; off > 0; off >>= 1) r += __shfl_xor(r, off);
        if (lane == 0) v[c] = r / (double)T;
    }
}

}  // namespace

int refine_chunk(int ncand, const int* nchans, const int* nsamp)
{
    int chunk = kChunk, most = 0;
    for (int b = 0; b < ncand; ++b) most = nchans[b] > most ? nchans[b] : most;
    auto items = [&] {
        long n = 0;
        for (int b = 0; b < ncand && n < 1024; ++b)
            n += (long)((nchans[b] + chunk - 1) / chunk) * ((nsamp[b] + kSeg - 1) / kSeg);
        return n;
    };
    while (chunk > kRefineChunkMin && chunk * chunk > 2 * most && items() < 1024) chunk /= 2;
    return chunk;
}

template <int NT>
static hipError_t launch_refine_passes(const refine_args& a, hipStream_t s)
{
    const dim3 items = linear_grid(a.nitems, kThreads);
    if (a.loss_kind == 1)
        hipLaunchKernelGGL(refine_power_kernel, linear_grid(a.ncand, 256, kPowerBlocksY), dim3(256), 0, s, a);
    for (int k0 = 0; k0 == 0 || k0 < a.scan_n; k0 += kScan) {
        const int nk = a.scan_n - k0 < kScan ? a.scan_n - k0 : kScan;
        if (nk > 0) {
            hipLaunchKernelGGL(refine_partial_kernel<kScan>, items, dim3(kThreads), 0, s, a, k0, nk);
            hipLaunchKernelGGL(refine_scan_loss_kernel<NT>, linear_grid(a.ncand, NT, nk), dim3(NT), 0, s, a, k0);
        }
        hipLaunchKernelGGL(refine_start_kernel, dim3(((unsigned)a.ncand + 63) / 64), dim3(64), 0, s, a, k0, nk);
    }
    for (int i = 0; i <= a.nsteps; ++i) {
        hipLaunchKernelGGL(refine_partial_kernel<0>, items, dim3(kThreads), 0, s, a, 0, 0);
        hipLaunchKernelGGL(refine_combine_kernel<NT>, linear_grid(a.ncand, NT), dim3(NT), 0, s, a, i == a.nsteps ? 1 : 0);
    }
    return hipGetLastError();
}

hipError_t launch_refine(const refine_args& a, hipStream_t s)
{
    if (a.ncand <= 0) return hipSuccess;
    if (a.nitems <= 0 || a.chunk < 1 || a.chunk > kChunk || (a.loss_kind != 0 && a.loss_kind != 1))
        return hipErrorInvalidValue;
    return a.longest <= 2 * kCombineShort ? launch_refine_passes<kCombineShort>(a, s)
                                          : launch_refine_passes<kCombineThreads>(a, s);
}

}  // namespace aa_hip

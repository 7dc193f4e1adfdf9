// First pass of the single-pulse search on one DM-time plane, the stage the
// reference's runner hands each range's device plane to
// (include/aa_permitted_pipelines_generic.hpp:848-889 -> analysis_GPU,
// src/aa_device_analysis.cu:126-133 reading [nDMs][nTimesamples]):
//
//  * boxcar MSD (the role of MSD_plane_profile, src/aa_device_MSD_plane_profile.cu):
//    mean and population sd of every in-row boxcar sum B_w(t) = sum_{i<w}
//    x[d][t+i], t + w <= nsamp, for w = 1..W (W <= 32), over the whole
//    plane.  Exact per width (the reference interpolates between decimated
//    widths).  One read of the plane.
//  * boxcar SNR (the first plane of SPDT, src/aa_device_SPS_long_kernel.cu:42-168):
//    snr[d][t] = max over widths that fit of (B_w(t) - mean_w) / sd_w and
//    width[d][t] = that w (ties: the smaller w; sd_w == 0 gives SNR 0).
//    One more read of the plane, one write of snr (float) and width (u16).
//
// Layout and numerics.  A tile is kTile consecutive start samples of one DM
// row plus the W-1 samples after them, staged in LDS.  Sums run in float on
// centred values (x - c), so a boxcar sum holds the noise and not the
// plane's offset: the MSD kernel centres each tile on its own mean, turns
// the tile's per-width float sums into (count, mean, centred second moment)
// in double and merges them into its workgroup's running moments with
// Chan's pairwise update (a persistent grid of kBlocks workgroups, tiles
// assigned by stride); one finalize workgroup merges the workgroups' moments
// in a fixed order, so the result does not depend on scheduling.  The SNR
// kernel centres on the plane mean c = mean_1 and divides
// (B'_w - (mean_w - w c)) by sd_w.
//
// Cost per start sample and width (W rounded up to 8, 16 or 32): 2 VALU
// operations in the MSD pass, 3.8 in the SNR pass.  Both passes read a run of
// consecutive start samples' samples into registers once (8 in the MSD pass, 4
// in the SNR pass).  Tiles at a row's end, where not every width fits, take 3
// and 5 operations and an LDS read.  VALU-bound at 32 widths; the plane is read
// twice from HBM.
//
// Measured on 1536 x 890,624 samples at W = 32 (2.4e9 instructions of a wave
// for the 2 and 3.8 operations, 7.1 ms at 4.34 cycles each and 2.4 GHz; 19.2 GB,
// 4.0 ms): MSD 2.76 ms, SNR 4.81 ms.  Before, MSD 4.77 ms: a third of its
// instructions were the sums over the lanes of 32 widths one at a time, the
// tile's staging (LDS written, read and written again to centre it) and one
// wave's serial sum over the tile's edges.  SNR 6.37 ms, with 5 operations per
// width and stores of one float at a stride of four.  Other limits, 512 x
// 200,000 samples, both passes: W = 5 1114 -> 326 us, 8 1186 -> 330, 16 1362 ->
// 380, 20 1466 -> 558.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <mutex>

#include "ddtr_kernels.h"

namespace aa_hip {
namespace {

constexpr int kThreads = 256;
constexpr int kK = 32;                    // start samples per thread per tile
constexpr int kTile = kThreads * kK;      // 8192 start samples of one row
constexpr int kMaxW = SPD_MAX_WIDTH;      // 32
constexpr int kBlocks = 1024;             // persistent MSD grid

struct spd_aux {              // finalize -> SNR kernel
    float c;                  // centring value: mean of width-1 sums (the plane mean)
    int finite;               // every off * rsd and rsd is
    float pad[2];
    float off[kMaxW];         // mean_w - w * c
    float rsd[kMaxW];         // 1 / sd_w (0 when sd_w == 0)
};

// v plus the value `ctrl` selects from another lane (DPP); lanes the row
// mask leaves out, or whose source is out of range, add 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v)
{
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}

// Sum over the wave's 64 lanes, in lane 63 only (other lanes hold partial
// sums): quad sums (quad_perm 1,0,3,2 then 2,3,0,1), row sums (row_shr 4
// then 8, lanes 12-15 of each row), then row_bcast15 and row_bcast31.  A
// fixed order of additions, in registers (no LDS traffic).
__device__ __forceinline__ float wave_sum_to_lane63(float v)
{
    v = dpp_add<0xB1, 0xf>(v);
    v = dpp_add<0x4E, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);
    v = dpp_add<0x143, 0xc>(v);
    return v;
}

// Sums over the wave's 64 lanes of N (32, 16 or 8) values, each lane keeping
// one: lane l gets value spread_width<N>(l)'s, of the lanes with the same value
// those without a bit of spread_again<N>() are one each.  Half of the values go
// to the other half of the lanes at each step (row swaps, then DPP with a
// select): at N = 32 70 instructions where a sum to lane 63 per value takes 21
// each.
template <int N>
__device__ __forceinline__ int spread_width(int lane)
{
    const int b5 = lane >> 5, b4 = lane >> 4 & 1, b3 = lane >> 3 & 1, b2 = lane >> 2 & 1, b1 = lane >> 1 & 1;
    return N == 32 ? b5 * 16 + b4 * 8 + b2 * 4 + b3 * 2 + b1 : N == 16 ? b5 * 8 + b4 * 4 + b2 * 2 + b3
                                                                      : b5 * 4 + b4 * 2 + b2;
}
template <int N>
constexpr int spread_again() { return N == 32 ? 1 : N == 16 ? 3 : 11; }
template <int CTRL>
__device__ __forceinline__ float spread_add(float a, float b, bool second)
{
    const float keep = second ? b : a, send = second ? a : b;
    return keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), CTRL, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float wave_spread_sum(const float (&a)[N], int lane)
{
    float v[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[i]), __float_as_uint(a[i + N / 2]), false, false);
        v[i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    }
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 4]), false, false);
        v[i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    }
    // row_ror:4 pairs lanes of unlike bit 2 (and any bit 3), row_ror:8 of unlike bit 3
#pragma unroll
    for (int i = 0; i < N / 8; ++i) v[i] = spread_add<0x124>(v[i], v[i + N / 8], lane & 4);
    if constexpr (N >= 16) {
#pragma unroll
        for (int i = 0; i < N / 16; ++i) v[i] = spread_add<0x128>(v[i], v[i + N / 16], lane & 8);
    } else {
        v[0] = dpp_add<0x128, 0xf>(v[0]);
    }
    v[0] = N == 32 ? spread_add<0x4E>(v[0], v[1], lane & 2) : dpp_add<0x4E, 0xf>(v[0]);
    return dpp_add<0xB1, 0xf>(v[0]);
}

// v plus the double `ctrl` selects from another lane of the row mask (0 from
// beyond the row).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_add64(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROW_MASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xf, false);
    return v + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Inclusive prefix sums over lanes 0-31.
__device__ __forceinline__ double scan32(double v)
{
    v = dpp_add64<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v = dpp_add64<0x112, 0xf>(v);
    v = dpp_add64<0x114, 0xf>(v);
    v = dpp_add64<0x118, 0xf>(v);
    return dpp_add64<0x142, 0xa>(v);   // row_bcast15
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4u __attribute__((aligned(4)));   // rows start at any float
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

// Chan et al.'s pairwise update: (n_a, m_a, M2_a) += (n_b, m_b, M2_b).
__device__ __forceinline__ void chan_merge(double& na, double& ma, double& m2a, double nb, double mb, double m2b)
{
    if (nb <= 0.0) return;
    const double n = na + nb;
    const double delta = mb - ma, part = nb / n;
    ma += delta * part;
    m2a += m2b + delta * delta * (na * part);
    na = n;
}

// Per-workgroup moments over its tiles: partial[blk][w] = (n_w, mean of B_w,
// sum of squared deviations of B_w).
// WC: the width limit W rounded up to 8, 16 or 32; widths past W are computed
// and left out.  EXACT: W is WC, known at compile time (a runtime limit costs a
// scalar condition per width in the tiles at a row's end, live across the loops:
// 8 % of the whole pass at 32).
// Four waves per SIMD (128 registers a lane): the persistent grid of
// kBlocks work-groups is resident at once only at four work-groups per CU.
template <int WC, bool EXACT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void spd_msd_kernel(
    const float* __restrict__ plane, long pitch, int ndms, int nsamp, int W_arg, double* __restrict__ partial)
{
    const int W = EXACT ? WC : W_arg;
    __shared__ __align__(16) float s[kTile + kMaxW];
    __shared__ float red[kThreads / 64][2 * kMaxW];
    __shared__ float wsum[kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const long per_row = ((long)nsamp + kTile - 1) / kTile;
    const long ntiles = (long)ndms * per_row;
    double accn = 0.0, accm = 0.0, acc2 = 0.0;   // thread tid < W: width tid + 1
    for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const long d = tile / per_row;
        const long t0 = (tile - d * per_row) * kTile;
        const float* row = plane + d * pitch;
        const long rest = (long)nsamp - t0;
        const int nout = (int)(rest < kTile ? rest : kTile);                 // start samples in the tile
        const int nload = (int)(rest < kTile + W - 1 ? rest : kTile + W - 1);  // samples staged
        // All WC widths fit at every start sample (a wave-uniform case).
        const bool fast = rest >= kTile + WC - 1;
        float c;
        if (fast) {
            // The tile waits in registers for its mean, so it is written to LDS
            // once and centred.
            f32x4 v[kK / 4];
#pragma unroll
            for (int k = 0; k < kK / 4; ++k)
                v[k] = *reinterpret_cast<const f32x4u*>(row + t0 + 4 * (tid + kThreads * k));
            const float after = tid < WC - 1 ? row[t0 + kTile + tid] : 0.0f;
            float part = 0.0f;
#pragma unroll
            for (int k = 0; k < kK / 4; ++k) part += (v[k].x + v[k].y) + (v[k].z + v[k].w);
            part = wave_sum_to_lane63(part);
            __syncthreads();   // the previous tile's readers of s, red and wsum are done
            if (lane == 63) wsum[wv] = part;
            __syncthreads();
            c = (wsum[0] + wsum[1] + wsum[2] + wsum[3]) / (float)nout;
#pragma unroll
            for (int k = 0; k < kK / 4; ++k) *reinterpret_cast<f32x4*>(s + 4 * (tid + kThreads * k)) = v[k] - c;
            if (tid < kMaxW) s[kTile + tid] = after - c;
            __syncthreads();
        } else {
            __syncthreads();   // the previous tile's readers of s, red and wsum are done
            float part = 0.0f;
            for (int i = tid; i < kTile + kMaxW; i += kThreads) {
                const float v = i < nload ? row[t0 + i] : 0.0f;
                s[i] = v;
                if (i < nout) part += v;
            }
            part = wave_sum_to_lane63(part);
            if (lane == 63) wsum[wv] = part;
            __syncthreads();
            c = (wsum[0] + wsum[1] + wsum[2] + wsum[3]) / (float)nout;
            for (int i = tid; i < nload; i += kThreads) s[i] -= c;
            __syncthreads();
        }
        float a1[WC], a2[WC];
#pragma unroll
        for (int w = 0; w < WC; ++w) a1[w] = a2[w] = 0.0f;
        // With all widths at every start sample the sums of B_w over the tile follow from the tile's sum C_0 and its
        // edges (below), so the loop keeps only the running sum and the
        // square sums; runs of kRun consecutive start samples per thread,
        // their kRun + 31 samples read once into registers with 16-byte
        // reads (instead of one LDS read per start sample and width).
        float cs = 0.0f;   // fast: this thread's part of C_0 = sum of s[0 .. kTile)
        if (fast) {
            constexpr int kRun = 8, kWin = kRun + WC;   // 40 registers: s[j0 .. j0 + 39]
            static_assert(kTile % (kRun * kThreads) == 0, "whole runs per thread");
#pragma unroll 1
            for (int k = 0; k < kTile / (kRun * kThreads); ++k) {
                const int j0 = kRun * (tid + kThreads * k);
                float v[kWin];
#pragma unroll
                for (int m = 0; m < kWin / 4; ++m) {
                    const float4 q = *reinterpret_cast<const float4*>(s + j0 + 4 * m);
                    v[4 * m] = q.x;
                    v[4 * m + 1] = q.y;
                    v[4 * m + 2] = q.z;
                    v[4 * m + 3] = q.w;
                }
#pragma unroll
                for (int i = 0; i < kRun; ++i) {
                    cs += v[i];
                    float B = 0.0f;
#pragma unroll
                    for (int w = 0; w < WC; ++w) {
                        B += v[i + w];
                        a2[w] = __builtin_fmaf(B, B, a2[w]);
                    }
                }
            }
        } else if (nload == kTile + W - 1) {   // every width fits at every start sample
#pragma unroll 2
            for (int k = 0; k < kK; ++k) {
                const int j = tid + kThreads * k;
                float B = 0.0f;
#pragma unroll
                for (int w = 0; w < WC; ++w) {
                    if (w < W) {
                        B += s[j + w];
                        a1[w] += B;
                        a2[w] = __builtin_fmaf(B, B, a2[w]);
                    }
                }
            }
        } else {   // the row's last tile: widths that fit
            for (int k = 0; k < kK; ++k) {
                const int j = tid + kThreads * k;
                if (j >= nout) break;
                float B = 0.0f;
#pragma unroll
                for (int w = 0; w < WC; ++w) {
                    if (w < W && j + w < nload) {
                        B += s[j + w];
                        a1[w] += B;
                        a2[w] = __builtin_fmaf(B, B, a2[w]);
                    }
                }
            }
        }
        const float r2 = wave_spread_sum(a2, lane);
        const float r1 = fast ? wave_sum_to_lane63(cs) : wave_spread_sum(a1, lane);
        const bool keeps = (lane & spread_again<WC>()) == 0;
        if (keeps) red[wv][kMaxW + spread_width<WC>(lane)] = r2;
        if (fast ? lane == 63 : keeps) red[wv][fast ? 0 : spread_width<WC>(lane)] = r1;
        __syncthreads();
        if (tid < W) {
            const int w = tid + 1;
            const int w1 = fast ? 0 : tid;
            double S1 = (double)red[0][w1] + (double)red[1][w1] + (double)red[2][w1] + (double)red[3][w1];
            if (fast) {
                // sum over the tile's starts j of B_w(j) = sum_{m<w} C_m, with
                // C_m = sum_{j<kTile} s[j + m] = C_{m-1} + s[kTile - 1 + m] - s[m - 1]
                const double e = tid > 0 ? (double)s[kTile - 1 + tid] - (double)s[tid - 1] : 0.0;
                S1 = scan32(S1 + scan32(e));
            }
            const double S2 = (double)red[0][kMaxW + tid] + (double)red[1][kMaxW + tid] +
                              (double)red[2][kMaxW + tid] + (double)red[3][kMaxW + tid];
            const long fit = (long)nload - w + 1;               // start samples whose width-w boxcar is staged
            const double n = (double)(fit < nout ? (fit > 0 ? fit : 0) : nout);
            if (n > 0.0) {   // the tile's moments of B_w = B'_w + w c
                const double mt = fast ? S1 * (1.0 / kTile) : S1 / n;
                const double m2t = S2 - S1 * mt;
                chan_merge(accn, accm, acc2, n, mt + (double)w * (double)c, m2t > 0.0 ? m2t : 0.0);
            }
        }
    }
    if (tid < W) {
        double* p = partial + ((long)blockIdx.x * kMaxW + tid) * 3;
        p[0] = accn;
        p[1] = accm;
        p[2] = acc2;
    }
}

// Merges the workgroups' moments in a fixed order; writes (mean_w, sd_w)
// and the SNR kernel's centring constants.  kFinLanes threads per width:
// lane i merges the partials of blocks i, i + kFinLanes, ... in turn, then
// the lanes' moments are merged pairwise in a fixed tree.
constexpr int kFinLanes = 32;
constexpr int kFinThreads = kMaxW * kFinLanes;
__global__ __launch_bounds__(kFinThreads) void spd_msd_finalize_kernel(const double* __restrict__ partial,
                                                                       int nblocks, int W, float* __restrict__ msd,
                                                                       spd_aux* __restrict__ aux)
{
    __shared__ double tn[kMaxW][kFinLanes], tm[kMaxW][kFinLanes], t2[kMaxW][kFinLanes];
    __shared__ double mean[kMaxW], sd[kMaxW];
    const int w = threadIdx.x / kFinLanes, i = threadIdx.x % kFinLanes;
    double n = 0.0, m = 0.0, m2 = 0.0;
    if (w < W)
        for (int b = i; b < nblocks; b += kFinLanes) {
            const double* p = partial + ((long)b * kMaxW + w) * 3;
            chan_merge(n, m, m2, p[0], p[1], p[2]);
        }
    tn[w][i] = n;
    tm[w][i] = m;
    t2[w][i] = m2;
    for (int h = kFinLanes / 2; h > 0; h >>= 1) {
        __syncthreads();
        if (i < h) {
            chan_merge(n, m, m2, tn[w][i + h], tm[w][i + h], t2[w][i + h]);
            tn[w][i] = n;
            tm[w][i] = m;
            t2[w][i] = m2;
        }
    }
    if (w < W && i == 0) {
        const double v = n > 0.0 ? m2 / n : 0.0;
        mean[w] = m;
        sd[w] = v > 0.0 ? sqrt(v) : 0.0;
        msd[2 * w] = (float)mean[w];
        msd[2 * w + 1] = (float)sd[w];
    }
    __syncthreads();
    bool finite = true;
    if (w < W && i == 0) {
        const double c = (double)(float)mean[0];
        const float off = (float)(mean[w] - (double)(w + 1) * c);
        const float rsd = sd[w] > 0.0 ? (float)(1.0 / sd[w]) : 0.0f;
        if (w == 0) aux->c = (float)c;
        aux->off[w] = off;
        aux->rsd[w] = rsd;
        finite = fabsf(rsd) < INFINITY && fabsf(off * rsd) < INFINITY;
    }
    finite = __syncthreads_and(finite);
    if (threadIdx.x == 0) aux->finite = finite;
}

template <int WC, bool EXACT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void spd_snr_kernel(
    const float* __restrict__ plane, long pitch, int nsamp, int W_arg, const spd_aux* __restrict__ aux,
    float* __restrict__ snr, long snr_pitch, uint16_t* __restrict__ width, long width_pitch)
{
    const int W = EXACT ? WC : W_arg;
    __shared__ __align__(16) float s[kTile + kMaxW];
    __shared__ float off[kMaxW];
    __shared__ __align__(16) float rsd[kMaxW], prod[kMaxW];   // prod: -off * rsd
    const int tid = threadIdx.x;
    const long per_row = ((long)nsamp + kTile - 1) / kTile;
    const long d = blockIdx.x / per_row;
    const long t0 = (blockIdx.x - d * per_row) * kTile;
    const float* row = plane + d * pitch;
    const long rest = (long)nsamp - t0;
    const int nout = (int)(rest < kTile ? rest : kTile);
    const int nload = (int)(rest < kTile + W - 1 ? rest : kTile + W - 1);
    const float c = aux->c;
    if (tid < kMaxW) {
        // widths past W: an SNR below every other
        off[tid] = tid < W ? aux->off[tid] : 0.0f;
        rsd[tid] = tid < W ? aux->rsd[tid] : 0.0f;
        prod[tid] = tid < W ? -off[tid] * rsd[tid] : -INFINITY;
    }
    const bool fast = rest >= kTile + WC - 1;   // all WC widths fit at every start sample
    if (fast) {
        f32x4 v[kK / 4];
#pragma unroll
        for (int k = 0; k < kK / 4; ++k)
            v[k] = *reinterpret_cast<const f32x4u*>(row + t0 + 4 * (tid + kThreads * k));
        const float after = tid < WC - 1 ? row[t0 + kTile + tid] : 0.0f;
#pragma unroll
        for (int k = 0; k < kK / 4; ++k) *reinterpret_cast<f32x4*>(s + 4 * (tid + kThreads * k)) = v[k] - c;
        if (tid < kMaxW) s[kTile + tid] = after - c;
    } else {
        for (int i = tid; i < kTile + kMaxW; i += kThreads) s[i] = i < nload ? row[t0 + i] - c : 0.0f;
    }
    __syncthreads();
    float* so = snr ? snr + d * snr_pitch + t0 : nullptr;
    uint16_t* wo = width ? width + d * width_pitch + t0 : nullptr;
    if (nload == kTile + W - 1) {   // every width fits at every start sample
        // SNR_w = B'_w * rsd_w - off_w * rsd_w: one FMA per width
        float p[WC], r[WC];
#pragma unroll
        for (int w = 0; w < WC; ++w) {
            r[w] = rsd[w];
            p[w] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(prod[w])));
        }
        // Finite: no SNR is a NaN (the offsets hold the plane's mean, so every
        // sample is finite as well), which the maxima below would pass over.
        if (fast && aux->finite) {
            // Runs of kRun consecutive start samples per thread, their
            // kRun + 31 samples read into registers once.  The largest SNR of
            // each kGroup widths is taken with max3; only the first group that
            // raised the maximum is kept, as its number and the boxcar sum
            // before it, and its SNRs are computed once more (the same
            // operations) to find the width: 3.8 operations per width where
            // keeping the width along with each maximum takes 5.
            constexpr int kRun = 4, kWin = kRun + WC;   // 36 registers: s[j0 .. j0 + 35]
            constexpr int kGroup = 4;
            static_assert(kTile % (kRun * kThreads) == 0, "whole runs per thread");
            const bool vec_s = so && ((uintptr_t)so & 15) == 0, vec_w = wo && ((uintptr_t)wo & 7) == 0;
#pragma unroll 1
            for (int k = 0; k < kTile / (kRun * kThreads); ++k) {
                const int j0 = kRun * (tid + kThreads * k);
                float v[kWin];
#pragma unroll
                for (int m = 0; m < kWin / 4; ++m) {
                    const float4 q = *reinterpret_cast<const float4*>(s + j0 + 4 * m);
                    v[4 * m] = q.x;
                    v[4 * m + 1] = q.y;
                    v[4 * m + 2] = q.z;
                    v[4 * m + 3] = q.w;
                }
                f32x4 best;
                u16x4 bw;
#pragma unroll
                for (int i = 0; i < kRun; ++i) {
                    float B = 0.0f, top = 0.0f, before = 0.0f;
                    int at = 0;   // first width - 1 of the group with the maximum
#pragma unroll
                    for (int g = 0; g < WC; g += kGroup) {
                        const float start = B;
                        float x[kGroup];
#pragma unroll
                        for (int w = 0; w < kGroup; ++w) {
                            B += v[i + g + w];
                            x[w] = __builtin_fmaf(B, r[g + w], p[g + w]);
                        }
                        float m = fmaxf(fmaxf(x[0], x[1]), x[2]);
                        if (g == 0) {
                            top = fmaxf(m, x[3]);
                        } else {
                            m = fmaxf(fmaxf(m, x[3]), top);
                            const bool more = m > top;
                            before = more ? start : before;
                            at = more ? g : at;
                            top = m;
                        }
                    }
                    const float* y = s + j0 + i + at;
                    const f32x4 rg = *reinterpret_cast<const f32x4*>(rsd + at);
                    const f32x4 pg = *reinterpret_cast<const f32x4*>(prod + at);
                    float x[kGroup];
#pragma unroll
                    for (int w = 0; w < kGroup; ++w) {
                        before += y[w];
                        x[w] = __builtin_fmaf(before, rg[w], pg[w]);
                    }
                    int n = 4;   // the first of the group that is the maximum
                    n = x[2] == top ? 3 : n;
                    n = x[1] == top ? 2 : n;
                    n = x[0] == top ? 1 : n;
                    best[i] = top;
                    bw[i] = (uint16_t)(at + n);
                }
                if (vec_s) {
                    *reinterpret_cast<f32x4*>(so + j0) = best;
                } else if (so) {
#pragma unroll
                    for (int i = 0; i < kRun; ++i) so[j0 + i] = best[i];
                }
                if (vec_w) {
                    *reinterpret_cast<u16x4*>(wo + j0) = bw;
                } else if (wo) {
#pragma unroll
                    for (int i = 0; i < kRun; ++i) wo[j0 + i] = bw[i];
                }
            }
            return;
        }
#pragma unroll 2
        for (int k = 0; k < kK; ++k) {
            const int j = tid + kThreads * k;
            float B = s[j];
            float best = __builtin_fmaf(B, r[0], p[0]);
            int bw = 1;
#pragma unroll
            for (int w = 1; w < WC; ++w) {
                if (w < W) {
                    B += s[j + w];
                    const float v = __builtin_fmaf(B, r[w], p[w]);
                    if (v > best) {
                        best = v;
                        bw = w + 1;
                    }
                }
            }
            if (so) so[j] = best;
            if (wo) wo[j] = (uint16_t)bw;
        }
        return;
    }
    for (int k = 0; k < kK; ++k) {
        const int j = tid + kThreads * k;
        if (j >= nout) break;
        float B = 0.0f, best = 0.0f;
        int bw = 0;
#pragma unroll
        for (int w = 0; w < kMaxW; ++w) {
            if (w < W && j + w < nload) {
                B += s[j + w];
                const float v = (B - off[w]) * rsd[w];
                if (bw == 0 || v > best) {
                    best = v;
                    bw = w + 1;
                }
            }
        }
        if (so) so[j] = best;
        if (wo) wo[j] = (uint16_t)bw;
    }
}

}  // namespace

size_t spd_workspace_bytes() { return (size_t)kBlocks * kMaxW * 3 * sizeof(double) + 256 + sizeof(spd_aux); }

hipError_t launch_spd_first_pass(const float* plane, size_t pitch, int ndms, int nsamp, int W, float* msd,
                                 float* snr, size_t snr_pitch, uint16_t* width, size_t width_pitch, void* work,
                                 hipStream_t s)
{
    if (!plane || !msd || !work || ndms <= 0 || nsamp <= 0 || W < 1 || W > kMaxW || W > nsamp ||
        pitch < (size_t)nsamp)
        return hipErrorInvalidValue;
    if ((snr && snr_pitch < (size_t)nsamp) || (width && width_pitch < (size_t)nsamp)) return hipErrorInvalidValue;
    double* partial = static_cast<double*>(work);
    spd_aux* aux = reinterpret_cast<spd_aux*>(static_cast<char*>(work) + (size_t)kBlocks * kMaxW * 3 * sizeof(double));
    const long per_row = ((long)nsamp + kTile - 1) / kTile;
    const long ntiles = (long)ndms * per_row;
    if (ntiles > 0x7fffffffL) return hipErrorInvalidValue;
#define AA_SPD_MSD(WC_, EXACT_) \
    hipLaunchKernelGGL((spd_msd_kernel<WC_, EXACT_>), dim3(kBlocks), dim3(kThreads), 0, s, plane, (long)pitch, ndms, nsamp, W, partial)
    if (W == kMaxW) AA_SPD_MSD(kMaxW, true);
    else if (W > 16) AA_SPD_MSD(kMaxW, false);
    else if (W == 16) AA_SPD_MSD(16, true);
    else if (W > 8) AA_SPD_MSD(16, false);
    else if (W == 8) AA_SPD_MSD(8, true);
    else AA_SPD_MSD(8, false);
#undef AA_SPD_MSD
    hipLaunchKernelGGL(spd_msd_finalize_kernel, dim3(1), dim3(kFinThreads), 0, s, (const double*)partial, kBlocks, W, msd, aux);
    if (snr || width) {
#define AA_SPD_SNR(WC_, EXACT_) \
    hipLaunchKernelGGL((spd_snr_kernel<WC_, EXACT_>), dim3((unsigned)ntiles), dim3(kThreads), 0, s, plane, (long)pitch, nsamp, W, \
                       (const spd_aux*)aux, snr, (long)snr_pitch, width, (long)width_pitch)
        if (W == kMaxW) AA_SPD_SNR(kMaxW, true);
        else if (W > 16) AA_SPD_SNR(kMaxW, false);
        else if (W == 16) AA_SPD_SNR(16, true);
        else if (W > 8) AA_SPD_SNR(16, false);
        else if (W == 8) AA_SPD_SNR(8, true);
        else AA_SPD_SNR(8, false);
#undef AA_SPD_SNR
    }
    return hipGetLastError();
}

// ------------------------------------------------ allocation-free variant
// Workspace of launch_spd_first_pass_static: a file-scope device array, one
// copy per device, held until the process ends.  The first pass needs the
// same fixed workspace for every plane (the persistent MSD grid's per-width
// moments and the finalize constants), so this size covers every call whose
// width limit is at most SPD_MAX_WIDTH.  Every byte a call reads is written
// earlier in the same call, so nothing needs clearing between calls.
constexpr size_t kSpdScratchBytes = (size_t)kBlocks * kMaxW * 3 * sizeof(double) + 256 + sizeof(spd_aux);
static __device__ __align__(256) unsigned char scratch[kSpdScratchBytes];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kScratchDevices] = {};   // device address of `scratch`, per device

// The current device's address of `scratch`, looked up once per device.
hipError_t scratch_address(void** out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}
}  // namespace

size_t spd_static_scratch_bytes() { return kSpdScratchBytes; }

hipError_t launch_spd_first_pass_static(const float* plane, size_t pitch, int ndms, int nsamp, int W, float* msd,
                                        float* snr, size_t snr_pitch, uint16_t* width, size_t width_pitch,
                                        hipStream_t s)
{
    if (spd_workspace_bytes() > kSpdScratchBytes) return hipErrorInvalidValue;
    void* work = nullptr;
    const hipError_t e = scratch_address(&work);
    if (e != hipSuccess) return e;
    return launch_spd_first_pass(plane, pitch, ndms, nsamp, W, msd, snr, snr_pitch, width, width_pitch, work, s);
}

}  // namespace aa_hip

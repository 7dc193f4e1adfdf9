// Zero-DM with outlier rejection on [t][c] samples, in place: the
// reference's zero_dm_outliers_kernel_channels
// (src/aa_device_zero_dm_outliers_kernel.cu:190-233, launched by
// src/aa_zero_dm_outliers.cpp:47-67 with 128 threads per time sample and
// outlier_sigma 3).  Per time sample:
//   1. mean and standard deviation over all channels;
//   2. up to 5 times: the same over the channels strictly inside
//      mean +- 3 sigma of the previous estimate, stopping once
//      old_mean - mean < 0.001 (signed, as written);
//   3. x' = (x - mean) + bandpass[c] in float, clamped to [0, 2^nbits - 1],
//      truncated; a NaN (no channel inside the limits) becomes 0.
// The statistics are the reference's streaming ones, and their rounding is
// kept: 128 accumulators (accumulator v takes channels v, v+128, ... in
// order; Initiate/Add_one at :15-29), merged pairwise (Merge at :31-40) as
// its block reduction does (v += v+64, v += v+32 for v < 64 and v < 32, then
// v += v+q for q = 16, 8, 4, 2, 1), then mean = M/j and stdev = sqrt(S/j)
// in double.  The operations mix float and double exactly as declared
// there; products feeding an add are fused (one rounding), which is how
// CUDA's default contraction compiles those lines.
//
// MI355X mapping: one wave per time sample.
//
// 8-bit rows of up to 8192 channels (outliers_u8_kernel): the row stays in
// registers.  M is an exact integer below 2^24 in every accumulator, so the
// mean depends on the selected values only, not on their order; and the only
// use of the standard deviation is to place two limits between integers.  So
// each pass sums the selected bytes, their squares and their number in
// integers, and takes the limits from the exact variance.  The reference's
// float S differs from the exact one by at most (ceil(nchans / 128) + 16) x
// 2^-24 of it (non-negative terms, one rounding per Add_one, two per Merge
// level, one in each difference); where a limit lies within (more than twice)
// that of an integer, the pass is repeated with the reference's own
// accumulators (a few rows in 1000 on noise).  Measured on 4096 channels x
// 262,144 samples of noise with 64 loud channels: 0.95 ms (2.3 TB/s; the
// accumulators in every pass took 4.7); bound by vector issue, 1360
// instructions a row (counted) at two thirds of the issue rate, the rest waits
// between dependent passes at 5 waves per SIMD (86 registers).
//
// Other rows (zero_dm_outliers_kernel: 16-bit samples, whose sums may round,
// and more channels) always run those accumulators: lane l holds accumulators
// l and l + 64 (so the first merge level is inside the lane and the rest are
// shuffles down to lane 0).  The 1/(j(j-1)) factors of Add_one are a table in
// LDS (correctly rounded doubles, the same values the division gives).
// Compute-bound on the float64 VALU (about 15 instructions per channel and
// pass, up to 6 passes); the row is re-read from L1/L2 for each pass, eight
// channels per lane at a time.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "ddtr_kernels.h"

namespace aa_hip {
namespace {

constexpr int kCoefTab = 256;   // Add_one factors for counts up to 255

struct welford {
    float M;
    float S;
    int j;
};

// SMALL: j * x and M stay below 2^24 (8-bit samples), so j * x - M, an
// integer, is exact in float and needs no float64 work.
template <bool SMALL>
__device__ __forceinline__ void wf_add(welford& a, float x, const double* coef)
{
    a.j += 1;
    const double rj = (double)a.j;
    a.M = a.M + x;
    const float ft = SMALL ? (float)a.j * x - a.M : (float)fma(rj, (double)x, -(double)a.M);
    const double c = a.j < kCoefTab ? coef[a.j] : 1.0 / (rj * (rj - 1.0));   // coef[1] = 0
    a.S = (float)fma(c * (double)ft, (double)ft, (double)a.S);
}

// Add_one on an empty accumulator with factor 0 (coef[1]) gives M = x,
// S = 0, j = 1 exactly, i.e. Initiate: one code path for every channel.
template <bool SMALL>
__device__ __forceinline__ void wf_push(welford& a, float x, const double* coef)
{
    wf_add<SMALL>(a, x, coef);
}

// a <- Merge(a, b), with the reference's handling of empty accumulators.
__device__ __forceinline__ void wf_merge(welford& a, float bM, float bS, int bj)
{
    if (bj <= 0) return;
    if (a.j == 0) {
        a.M = bM;
        a.S = bS;
        a.j = bj;
        return;
    }
    const double rb = (double)bj, ra = (double)a.j;
    const float ft = (float)fma(rb / ra, (double)a.M, -(double)bM);
    const double coef = ra / (rb * (ra + rb));
    a.S = (float)fma(coef * (double)ft, (double)ft, (double)(a.S + bS));
    a.M = a.M + bM;
    a.j += bj;
}

// Lane 0's reduction of the wave's 128 accumulators, broadcast: mean, stdev.
__device__ __forceinline__ void wf_reduce(welford v0, const welford& v1, int lane, float& mean, float& stdev)
{
    wf_merge(v0, v1.M, v1.S, v1.j);   // accumulator l += l + 64
#pragma unroll
    for (int q = 32; q > 0; q >>= 1) {
        const float bM = __shfl_down(v0.M, q);
        const float bS = __shfl_down(v0.S, q);
        const int bj = __shfl_down(v0.j, q);
        if (lane < q) wf_merge(v0, bM, bS, bj);
    }
    float m = 0.0f, s = 0.0f;
    if (lane == 0) {
        m = (float)((double)v0.M / (double)v0.j);
        s = (float)sqrt((double)v0.S / (double)v0.j);
    }
    mean = __shfl(m, 0);
    stdev = __shfl(s, 0);
}

// Statistics of the row's channels strictly inside (lo, hi), as the
// reference accumulates them.  Channels come in batches of 8 per lane
// (lane + 64 k), all loads issued before the first add.
template <class T, bool SMALL>
__device__ __forceinline__ void wf_row(const T* row, int nchans, int lane, float lo, float hi, const double* coef,
                                       float& mean, float& stdev)
{
    welford v0{0.0f, 0.0f, 0}, v1{0.0f, 0.0f, 0};
    for (int c = lane; c < nchans; c += 512) {
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = c + 64 * k < nchans ? (float)row[c + 64 * k] : NAN;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (x[k] > lo && x[k] < hi) wf_push<SMALL>((k & 1) ? v1 : v0, x[k], coef);
    }
    wf_reduce(v0, v1, lane, mean, stdev);
}

__device__ __forceinline__ float outlier_value(float x, float mean, float bp, float maxval)
{
    return fminf(fmaxf((x - mean) + bp, 0.0f), maxval);   // fmaxf(NaN, 0) = 0
}

template <class T, bool SMALL>
__global__ __launch_bounds__(256) void zero_dm_outliers_kernel(T* data, long nsamp, int nchans,
                                                               const float* __restrict__ bp, float maxval)
{
    __shared__ double coef[kCoefTab];
    for (int i = threadIdx.x; i < kCoefTab; i += 256)
        coef[i] = i >= 2 ? 1.0 / ((double)i * ((double)i - 1.0)) : 0.0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const long waves = (long)gridDim.x * 4;
    for (long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6); t < nsamp; t += waves) {
        T* row = data + t * (long)nchans;
        float mean = 0.0f, stdev = 0.0f;
        // Pass 0 takes every channel (limits -inf, +inf); then up to 5
        // rejection passes.
        float lo = -INFINITY, hi = INFINITY;
        for (int f = 0; f < 6; ++f) {
            const float old_mean = mean;
            wf_row<T, SMALL>(row, nchans, lane, lo, hi, coef, mean, stdev);
            if (f > 0 && old_mean - mean < 0.001f) break;   // wave-uniform
            lo = fmaf(-3.0f, stdev, mean);
            hi = fmaf(3.0f, stdev, mean);
        }
        for (int c = lane; c < nchans; c += 64)
            row[c] = (T)(uint32_t)outlier_value((float)row[c], mean, bp[c], maxval);
    }
}

constexpr int kOutMaxChans = 8192;   // outliers_u8_kernel: 8 quads of 16 channels per lane

typedef uint32_t u32x4o __attribute__((ext_vector_type(4)));

// Sum over the wave, in every lane.
__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);    // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);    // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);    // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);    // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane(x, 63);
}

// 16 channels of a row from channel c, zero past the row.  TAIL: nchans is no
// multiple of 16; its last quad is read and written in pieces of 8, 4, 2 and 1.
template <bool TAIL>
__device__ __forceinline__ u32x4o load_quad(const uint8_t* row, int nchans, int c)
{
    u32x4o v = {0, 0, 0, 0};
    if (c + 16 <= nchans) {
        __builtin_memcpy(&v, row + c, 16);
    } else if (TAIL && c < nchans) {
        const int rem = nchans & 15;   // wave-uniform
        const uint8_t* p = row + c;
        if (rem & 8) __builtin_memcpy(&v, p, 8);
        if (rem & 4) {
            uint32_t w;
            __builtin_memcpy(&w, p + (rem & 8), 4);
            if (rem & 8) v[2] = w;
            else v[0] = w;
        }
        uint32_t last = 0;   // the dword of the last 1 to 3 bytes
        if (rem & 2) {
            uint16_t w;
            __builtin_memcpy(&w, p + (rem & 12), 2);
            last = w;
        }
        if (rem & 1) last |= (uint32_t)p[rem & 14] << (8 * (rem & 2));
        switch (rem >> 2) {
            case 0: v[0] |= last; break;
            case 1: v[1] |= last; break;
            case 2: v[2] |= last; break;
            default: v[3] |= last; break;
        }
    }
    return v;
}

template <bool TAIL>
__device__ __forceinline__ void store_quad(uint8_t* row, int nchans, int c, u32x4o v)
{
    if (c + 16 <= nchans) {
        __builtin_memcpy(row + c, &v, 16);
    } else if (TAIL && c < nchans) {
        const int rem = nchans & 15;
        uint8_t* p = row + c;
        if (rem & 8) __builtin_memcpy(p, &v, 8);
        if (rem & 4) {
            const uint32_t w = (rem & 8) ? v[2] : v[0];
            __builtin_memcpy(p + (rem & 8), &w, 4);
        }
        const uint32_t last = (rem >> 2) == 0 ? v[0] : (rem >> 2) == 1 ? v[1] : (rem >> 2) == 2 ? v[2] : v[3];
        if (rem & 2) {
            const uint16_t w = (uint16_t)last;
            __builtin_memcpy(p + (rem & 12), &w, 2);
        }
        if (rem & 1) p[rem & 14] = (uint8_t)(last >> (8 * (rem & 2)));
    }
}

template <int NQ, bool TAIL>
__global__ __launch_bounds__(256) void outliers_u8_kernel(uint8_t* data, long nsamp, int nchans,
                                                          const float* __restrict__ bp, float maxval)
{
    __shared__ double coef[kCoefTab];
    extern __shared__ float bpl[];   // bandpass, zero past the channels
    for (int i = threadIdx.x; i < kCoefTab; i += 256)
        coef[i] = i >= 2 ? 1.0 / ((double)i * ((double)i - 1.0)) : 0.0;
    for (int i = threadIdx.x; i < NQ * 1024; i += 256) bpl[i] = i < nchans ? bp[i] : 0.0f;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const long waves = (long)gridDim.x * 4;
    long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= nsamp) return;   // no barrier below
    const uint32_t pad = (uint32_t)(NQ * 1024 - nchans);   // zero bytes counted as channels
    const float slack = (float)((nchans + 127) / 128 + 32) * 0x1p-24f;   // of sigma; twice the bound above and more
    u32x4o next[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) next[k] = load_quad<TAIL>(data + t * nchans, nchans, 16 * (64 * k + lane));
    for (; t < nsamp; t += waves) {
        uint8_t* row = data + t * (long)nchans;
        u32x4o q[NQ];
#pragma unroll
        for (int k = 0; k < NQ; ++k) q[k] = next[k];
        const long tn = t + waves < nsamp ? t + waves : t;
#pragma unroll
        for (int k = 0; k < NQ; ++k) next[k] = load_quad<TAIL>(data + tn * nchans, nchans, 16 * (64 * k + lane));

        int a = 0, b = 255;   // the selected values
        float mean = 0.0f;
        for (int f = 0; f < 6; ++f) {
            // sum, sum of squares and number of the selected bytes
            uint32_t m = 0, m2 = 0, n = 0;
            if (a == 0 && b == 255) {
#pragma unroll
                for (int k = 0; k < NQ; ++k)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        m = __builtin_amdgcn_udot4(q[k][i], 0x01010101u, m, false);
                        m2 = __builtin_amdgcn_udot4(q[k][i], q[k][i], m2, false);
                    }
                n = (uint32_t)nchans;
            } else {
                // bit 7 of the average of x and 256 - v is x >= v; v = 0 is
                // always true, v = 256 never
                const uint32_t ya = a > 0 ? (uint32_t)(256 - a) * 0x01010101u : 0u;
                const uint32_t yb = b < 255 ? (uint32_t)(255 - b) * 0x01010101u : 0u;
                const uint32_t all = a > 0 ? 0u : 0x80808080u;
#pragma unroll
                for (int k = 0; k < NQ; ++k)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t x = q[k][i];
                        const uint32_t ge = __builtin_amdgcn_lerp(x, ya, 0u) | all;
                        const uint32_t in = ge & ~__builtin_amdgcn_lerp(x, yb, 0u) & 0x80808080u;
                        const uint32_t xs = x & ((in - (in >> 7)) | in);
                        n += (uint32_t)__popc(in);
                        m = __builtin_amdgcn_udot4(xs, 0x01010101u, m, false);
                        m2 = __builtin_amdgcn_udot4(xs, xs, m2, false);
                    }
                n = wave_sum(n);
                if (a == 0) n -= pad;
            }
            m = wave_sum(m);
            m2 = wave_sum(m2);
            const float old_mean = mean;
            mean = (float)((double)m / (double)n);   // NaN for an empty selection, as 0 / 0
            if (f > 0 && old_mean - mean < 0.001f) break;   // wave-uniform
            if (n == 0 || f == 5) break;                    // stays NaN; the last pass
            // limits: mean -+ 3 sigma, sigma from the exact variance
            const double var = ((double)m2 * (double)n - (double)m * (double)m) / ((double)n * (double)n);
            const float sd = sqrtf((float)var);
            float lo = mean - 3.0f * sd, hi = mean + 3.0f * sd;
            const float d = 3.0f * sd * slack + 4e-5f;   // and the rounding of values below 256
            // a limit near no integer of 0..255 selects the same values as the
            // reference's
            const float rl = rintf(lo), rh = rintf(hi);
            if ((fabsf(lo - rl) <= d && rl >= 0.0f && rl <= 255.0f) ||
                (fabsf(hi - rh) <= d && rh >= 0.0f && rh <= 255.0f)) {
                float em, es;
                wf_row<uint8_t, true>(row, nchans, lane, (float)a - 0.5f, (float)b + 0.5f, coef, em, es);
                lo = fmaf(-3.0f, es, mean);
                hi = fmaf(3.0f, es, mean);
            }
            const int na = (int)fminf(fmaxf(floorf(lo) + 1.0f, 0.0f), 256.0f);
            const int nb = (int)fmaxf(fminf(ceilf(hi) - 1.0f, 255.0f), -1.0f);
            if (na == a && nb == b) break;   // the same values again: the same mean
            a = na;
            b = nb;
            if (a > b) {   // no value left
                mean = NAN;
                break;
            }
        }
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            const int c = 16 * (64 * k + lane);
            u32x4o o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 w = *reinterpret_cast<const float4*>(bpl + c + 4 * i);
                const uint32_t x = q[k][i];
                const uint32_t y0 = (uint32_t)outlier_value((float)(x & 0xffu), mean, w.x, maxval);
                const uint32_t y1 = (uint32_t)outlier_value((float)((x >> 8) & 0xffu), mean, w.y, maxval);
                const uint32_t y2 = (uint32_t)outlier_value((float)((x >> 16) & 0xffu), mean, w.z, maxval);
                const uint32_t y3 = (uint32_t)outlier_value((float)(x >> 24), mean, w.w, maxval);
                o[i] = y0 | y1 << 8 | y2 << 16 | y3 << 24;
            }
            store_quad<TAIL>(row, nchans, c, o);
        }
    }
}

template <int NQ>
void launch_outliers_u8(uint8_t* data, long nsamp, int nchans, const float* bp, float maxval, hipStream_t s)
{
    const long blocks = (nsamp + 3) / 4;
    const dim3 grid((unsigned)(blocks < 2048 ? blocks : 2048));
    const size_t lds = (size_t)NQ * 1024 * sizeof(float);
    if (nchans % 16 == 0)
        hipLaunchKernelGGL((outliers_u8_kernel<NQ, false>), grid, dim3(256), lds, s, data, nsamp, nchans, bp, maxval);
    else
        hipLaunchKernelGGL((outliers_u8_kernel<NQ, true>), grid, dim3(256), lds, s, data, nsamp, nchans, bp, maxval);
}

template <class T>
hipError_t launch_outliers(T* data, long nsamp, int nchans, const float* bp, int nbits, hipStream_t s)
{
    if (!data || !bp || nsamp < 0 || nchans <= 0 || nbits < 1 || nbits > 16) return hipErrorInvalidValue;
    if (nsamp == 0) return hipSuccess;
    const long blocks = (nsamp + 3) / 4;
    const unsigned grid = (unsigned)(blocks < 16384 ? blocks : 16384);
    const float maxval = (float)((1u << nbits) - 1u);
    if (sizeof(T) == 1 && nchans <= kOutMaxChans) {
        uint8_t* d = reinterpret_cast<uint8_t*>(data);
        if (nchans <= 1024) launch_outliers_u8<1>(d, nsamp, nchans, bp, maxval, s);
        else if (nchans <= 2048) launch_outliers_u8<2>(d, nsamp, nchans, bp, maxval, s);
        else if (nchans <= 4096) launch_outliers_u8<4>(d, nsamp, nchans, bp, maxval, s);
        else launch_outliers_u8<8>(d, nsamp, nchans, bp, maxval, s);
        return hipGetLastError();
    }
    // Counts per accumulator reach ceil(nchans / 128); with 8-bit samples
    // j * x and M stay below 2^24 while that count stays below 65793.
    const bool small = sizeof(T) == 1 && (nchans + 127) / 128 < 65793;
    if (small)
        hipLaunchKernelGGL((zero_dm_outliers_kernel<T, true>), dim3(grid), dim3(256), 0, s, data, nsamp, nchans, bp,
                           maxval);
    else
        hipLaunchKernelGGL((zero_dm_outliers_kernel<T, false>), dim3(grid), dim3(256), 0, s, data, nsamp, nchans,
                           bp, maxval);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_zero_dm_outliers_u8(uint8_t* data_tc, long nsamp, int nchans, const float* bp, int nbits,
                                      hipStream_t s)
{
    if (nbits > 8) return hipErrorInvalidValue;
    return launch_outliers<uint8_t>(data_tc, nsamp, nchans, bp, nbits, s);
}

hipError_t launch_zero_dm_outliers_u16(uint16_t* data_tc, long nsamp, int nchans, const float* bp, int nbits,
                                       hipStream_t s)
{
    return launch_outliers<uint16_t>(data_tc, nsamp, nchans, bp, nbits, s);
}

}  // namespace aa_hip

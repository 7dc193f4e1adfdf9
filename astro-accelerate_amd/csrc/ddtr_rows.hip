// Dedispersion of small ranges straight from the u8 rows, for gfx950.
//
// The LDS and matrix kernels share rows between 16 DM trials: a work-group
// fills a CU, its tile is 1000 to 2000 samples of 16 trials, and its channels
// follow one another behind a barrier each.  A small range leaves most of the
// chip idle that way and takes one tile's time, 25 to 30 us at 128 channels.
// Here a work-group is one trial's 1008 samples, so the same range is hundreds
// of work-groups of 4 waves, and nothing is staged: wave w sums a quarter of
// the channels, each lane 16 samples of them.
//
// Per channel a lane loads the 16 bytes from a whole dword on (loads at odd
// bytes run at a quarter of the rate), takes the next dword from lane + 1, and
// shifts the bytes left over out in registers; lane 63 only feeds lane 62.  The
// delays of 64 channels are computed at once, one per lane, and read back as
// scalars, so the loads of 8 channels are in flight together.  Sums are 16-bit
// pairs: whole dwords are added as pairs (even + 256 odd), the odd bytes apart,
// and the even sums follow at the end modulo 2^16; 256 channels of 255 fit.
//
// Bound: latency at the smallest sizes, then the vector memory path (a byte
// from L2 per add) and the 23 instructions per 16 adds and lane: 22 to 25 T
// adds/s.  Sharing rows pays from there on, unless the trials are so far apart
// that the shared windows are mostly unused, or too wide for LDS: then the byte
// row shapes run at 8 to 20 T adds/s and the direct kernel at 1.4.
//
// Measured, whole chunks with their corner turn: 128 channels x 16,384 samples,
// 128 and 64 trials 67.5 -> 27.6 us; 64 x 4032 samples of 128 channels 57 -> 13
// us; 64 trials 11 DM units apart x 30,240 samples of 640 channels 810 -> 90 us,
// x 55,328 of 2400 channels 5.76 -> 0.63 ms.
#include "ddtr_rows.h"

#include <cmath>

#include "linear_grid.h"

namespace aa_hip {

namespace {

constexpr int kRowWaves = 4;
constexpr int kRowThreads = 64 * kRowWaves;
constexpr int kRowTile = 63 * 16;                 // samples per work-group
constexpr int kRowChannels = 256 * kRowWaves;     // 16-bit sums per wave

typedef uint32_t u32x4r __attribute__((ext_vector_type(4)));
typedef u32x4r u32x4w __attribute__((aligned(4)));   // 16 bytes at a whole dword
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

struct row_sums {
    u16x2 all[4];       // per dword: even bytes + 256 odd bytes, modulo 2^16
    uint32_t odd[4];    // odd bytes, two 16-bit sums
};

__device__ __forceinline__ void row_add(u32x4r v, uint32_t shift, row_sums& a)
{
    uint32_t R[5];
#pragma unroll
    for (int k = 0; k < 4; ++k) R[k] = v[k];
    R[4] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)R[0], 0x130, 0xf, 0xf, true);   // wave_shl:1
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t x = __builtin_amdgcn_alignbyte(R[k + 1], R[k], shift);
        a.all[k] += __builtin_bit_cast(u16x2, x);
        a.odd[k] += (x >> 8) & 0x00ff00ffu;
    }
}

__global__ __launch_bounds__(kRowThreads) void dedisperse_rows_kernel(lds_params p)
{
    __shared__ __align__(16) uint32_t part[kRowWaves][64 * 8];   // 16-bit sums, two samples per dword
    // Work-group g runs on XCD g % 8: each XCD takes a run of consecutive
    // tiles, DM trials of one time tile after another, which share their rows.
    const int n_t = (p.t_processed + kRowTile - 1) / kRowTile;
    const int ntiles = p.ndms * n_t;
    const int per = (ntiles + 7) / 8;
    const int g = (int)linear_block();
    const int tile = (g & 7) * per + (g >> 3);
    if ((g >> 3) >= per || tile >= ntiles) return;   // whole work-group, before the barrier
    const int d = tile % p.ndms;
    const long t0 = (long)(tile / p.ndms) * kRowTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const float shift_temp = __fmaf_rn((float)d, p.mdmstep, p.mstartdm);
    const uint8_t* __restrict__ rows = p.L + t0;
    uint32_t s[4] = {0u, 0u, 0u, 0u};
    for (int b0 = 0; b0 < p.nchans; b0 += kRowChannels) {
        const int left = p.nchans - b0 < kRowChannels ? p.nchans - b0 : kRowChannels;
        const int end = b0 + left * (wave + 1) / kRowWaves;
        row_sums a;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            a.all[k] = u16x2{0, 0};
            a.odd[k] = 0u;
        }
        for (int c0 = b0 + left * wave / kRowWaves; c0 < end; c0 += 64) {
            const int n = end - c0 < 64 ? end - c0 : 64;
            const int delays = lane < n ? (int)__fmul_rn(p.dmshifts[c0 + lane], shift_temp) : 0;
            const uint8_t* row = rows + (size_t)c0 * p.pitch;
            int i = 0;
            for (; i + 8 <= n; i += 8) {
                u32x4r v[8];
                int delay[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    delay[j] = __builtin_amdgcn_readlane(delays, i + j);
                    v[j] = *reinterpret_cast<const u32x4w*>(row + (size_t)(delay[j] & ~3) + 16 * lane);
                    row += p.pitch;
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) row_add(v[j], (uint32_t)delay[j] & 3u, a);
            }
            for (; i < n; ++i, row += p.pitch) {
                const int delay = __builtin_amdgcn_readlane(delays, i);
                row_add(*reinterpret_cast<const u32x4w*>(row + (size_t)(delay & ~3) + 16 * lane), (uint32_t)delay & 3u,
                        a);
            }
        }
        if (b0 > 0) __syncthreads();   // the sums before these have been read
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4r o;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u16x2 odd = __builtin_bit_cast(u16x2, a.odd[2 * h + k]);
                const u16x2 even = a.all[2 * h + k] - (odd << 8);
                o[2 * k] = (uint32_t)even.x | (uint32_t)odd.x << 16;
                o[2 * k + 1] = (uint32_t)even.y | (uint32_t)odd.y << 16;
            }
            *reinterpret_cast<u32x4r*>(&part[wave][8 * lane + 4 * h]) = o;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w) {   // samples 4 threadIdx.x .. + 3
            const uint2 x = *reinterpret_cast<const uint2*>(&part[w][2 * threadIdx.x]);
            s[0] += x.x & 0xffffu;
            s[1] += x.x >> 16;
            s[2] += x.y & 0xffffu;
            s[3] += x.y >> 16;
        }
    }
    if (threadIdx.x >= kRowTile / 4) return;
    float* orow = p.out + (size_t)d * p.out_pitch;
    store_out4(orow, t0 + 4 * (long)threadIdx.x, p.t_processed, (reinterpret_cast<uintptr_t>(orow) & 15u) == 0,
               out_values4(s, p));
}

}  // namespace

// Time model behind the choice, in us, from plans of 32 to 1024 channels with
// fine and coarse DM steps: this kernel 22 to 25 T adds/s on top of 3 us and
// 1.2 ns per work-group; the others a tile at a time per CU, 8 us to start and
// end it.
namespace {

double rows_us(int nchans, int ndms, int t_processed)
{
    return 3.0 + (double)nchans * ndms * t_processed / 23e6 + 1.2e-3 * ndms * (t_processed / kRowTile + 1);
}

double tiles_us(double tiles, double tile_us)
{
    const double rounds = tiles / 256.0;   // one tile per CU at a time; few rounds end together
    return tile_us * (rounds < 2.0 ? (rounds <= 1.0 ? 1.0 : 2.0) : rounds);
}

}  // namespace

bool rows_beat_matrix(int nchans, int ndms, int t_processed, const matrix_layout& lay)
{
    const double tiles = (double)lay.n_dm_tiles * ((t_processed + lay.tile_out - 1) / lay.tile_out);
    return rows_us(nchans, ndms, t_processed) < 0.9 * tiles_us(tiles, 8.0 + 0.62 * lay.tile_cost);
}

// Tiles of a range in chunk shape `variant`, and the time of one.
static double shape_tiles(int nchans, int ndms, int t_processed, int variant, double* tile_us)
{
    static const double rate[kLdsVariants] = {21, 19, 38, 21, 47, 44, 33};   // T adds/s, all CUs busy
    const double samples = (double)lds_tile_samples(variant), dms = lds_tile_dms(variant);
    *tile_us = 8.0 + nchans * samples * dms * 256.0 / (rate[variant] * 1e6);
    return std::ceil(ndms / dms) * std::ceil(t_processed / samples);
}

bool rows_beat_shape(int nchans, int ndms, int t_processed, int variant)
{
    if (variant < 0) return true;   // the direct kernel: 1.4 T adds/s
    double tile_us;
    const double tiles = shape_tiles(nchans, ndms, t_processed, variant, &tile_us);
    return rows_us(nchans, ndms, t_processed) < 0.9 * tiles_us(tiles, tile_us);
}

// The matrix launch pays for its last round of tiles, the shared one does not.
// Measured on 150 batches of 4 and 16 equal beams (64 to 1024 channels, 536 to
// 2144 tiles a range): with this rule no batch is slower than with all ranges in
// shared launches, and those left there would gain 11 % at most; from 512 tiles
// on whatever the channels, 16 beams of 64 channels x 512 trials x 30,000 samples
// took 755 us against 601, of 192 channels at coarse steps 2259 against 1802.
bool matrix_beats_shared(int nchans, int ndms, int t_processed, const matrix_layout& lay, int variant)
{
    if (variant < 0) return true;   // it would run a launch of its own anyway
    const double rounds = (double)lay.n_dm_tiles * ((t_processed + lay.tile_out - 1) / lay.tile_out) / 256.0;
    const double matrix = (rounds < 4.0 ? std::ceil(rounds) : rounds + 0.5) * (8.0 + 0.62 * lay.tile_cost);
    double tile_us;
    const double tiles = shape_tiles(nchans, ndms, t_processed, variant, &tile_us);
    return matrix < 0.92 * tile_us * tiles / 256.0;
}

hipError_t launch_dedisperse_rows(const lds_params& p, hipStream_t s)
{
    if (!p.L || !p.dmshifts || !p.out || p.nchans <= 0 || (uintptr_t)p.L % 4 != 0 ||
        p.pitch % 4 != 0)
        return hipErrorInvalidValue;
    if (p.ndms <= 0 || p.t_processed <= 0) return hipSuccess;
    const long tiles = (long)p.ndms * ((p.t_processed + kRowTile - 1) / kRowTile);
    if (tiles > 0x0fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(dedisperse_rows_kernel, linear_grid(8 * ((tiles + 7) / 8), kRowThreads), dim3(kRowThreads), 0, s,
                       p);
    return hipGetLastError();
}

}  // namespace aa_hip

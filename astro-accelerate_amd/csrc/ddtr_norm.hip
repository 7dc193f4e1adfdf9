// Column normalisation of a [rows][cols] array in place: the reference's
// normalization_transposed_kernel (src/aa_device_zero_dm_kernel.cu:100-164),
// which both DDTR normalisation options run:
//   - input normalisation on each [t][c] chunk before its corner turn, with
//     cols = nchans and factor (2^nbits - 1)/2 (src/aa_zero_dm.cpp:49-60,
//     called at include/aa_permitted_pipelines_generic.hpp:731-735);
//   - output normalisation on each [dm][t] plane, with cols = t_processed
//     and factor 127.5 (src/aa_zero_dm.cpp:62-74, called at
//     include/aa_permitted_pipelines_generic.hpp:823-831).
// Per column: 32 float partial sums, partial y adding rows y, y+32, ... in
// row order; then p[y] += p[y+i] for i = 16, 8, 4, 2, 1; s = p[0]/rows -
// factor; every value becomes x - s (integers: clamped to [0, 2^nbits - 1]
// and truncated).  The float sums round, so the order is kept exactly:
//   - normalize_strip_f32_kernel (float planes of at most 1536 rows; 64 or 16
//     columns per workgroup) keeps each partial in its own lanes and the strip
//     in registers between the sums and the write: one read, one write.  1536
//     rows are 48 float4 per lane: 216 of the 256 registers that two waves per
//     SIMD leave a lane.
//   - normalize_columns_kernel keeps it literally (64 columns per
//     workgroup, wave w owns partials w and w + 16), with a second read to
//     apply.  It serves taller float planes (wide ones at 4 columns per lane,
//     normalize_columns_f32x4_kernel) and any integer data.
//   - For integer data whose partial sums cannot pass 2^24
//     (ceil(rows/32) * type max <= 2^24, e.g. u8 chunks up to 2,105,376
//     rows), every float partial is an exact integer, so the tall input
//     chunks are summed in integers over row segments spread across the
//     chip (atomic adds into 32 x cols counters), and only the tree runs in
//     float.  Same result, many more workgroups.
// HBM-bound.  Measured, before with two reads of a float plane and lanes
// numbered along one row of 16-byte words: a 1536 x 222,656 float plane 0.87 ->
// 0.56 ms (4.9 TB/s of one read and one write), 262,144 u8 rows x 4096 0.82 ->
// 0.65 ms (5.0 TB/s of two reads and a write), x 384 191 -> 75 us, x 16 170 ->
// 36 us (the rest: scratch allocation and five launches).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "ddtr_kernels.h"
#include "linear_grid.h"

namespace aa_hip {
namespace {

__device__ __forceinline__ float norm_value(float x, float s, float maxval)
{
    float r = __fsub_rn(x, s);
    return r < 0.0f ? 0.0f : (r > maxval ? maxval : r);
}

// The 16-8-4-2-1 tree over p[0..15] (p[y] already holds partials y + y+16)
// and the column offset s.
__device__ __forceinline__ float norm_offset(float (&p)[16], long rows, float factor)
{
#pragma unroll
    for (int i = 8; i > 0; i >>= 1)
#pragma unroll
        for (int y = 0; y < i; ++y) p[y] = __fadd_rn(p[y], p[y + i]);
    return __fsub_rn(__fdiv_rn(p[0], (float)rows), factor);
}

template <class T>
__global__ __launch_bounds__(1024) void normalize_columns_kernel(T* data, long rows, long cols, float factor,
                                                                 float maxval)
{
    __shared__ float part[16][64];
    __shared__ float offs[64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long c = linear_block() * 64 + lane;
    const bool on = c < cols;
    float a0 = 0.0f, a1 = 0.0f;
    if (on) {
#pragma unroll 4
        for (long r = w; r < rows; r += 32) {
            a0 = __fadd_rn(a0, (float)data[r * cols + c]);
            if (r + 16 < rows) a1 = __fadd_rn(a1, (float)data[(r + 16) * cols + c]);
        }
    }
    part[w][lane] = __fadd_rn(a0, a1);
    __syncthreads();
    if (w == 0) {
        float p[16];
#pragma unroll
        for (int y = 0; y < 16; ++y) p[y] = part[y][lane];
        offs[lane] = norm_offset(p, rows, factor);
    }
    __syncthreads();
    if (!on) return;
    const float s = offs[lane];
    for (long r = w; r < rows; r += 16) {
        T* v = data + r * cols + c;
        if constexpr (std::is_same<T, float>::value)
            *v = __fsub_rn(*v, s);
        else
            *v = (T)(uint32_t)norm_value((float)*v, s, maxval);
    }
}

// Wide float planes of a multiple of 4 columns: the same order, 4 columns per
// lane (16-byte accesses), 256 columns per workgroup.
__global__ __launch_bounds__(1024) void normalize_columns_f32x4_kernel(float* data, long rows, long cols,
                                                                       float factor)
{
    __shared__ float4 part[16][64];
    __shared__ float4 offs[64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long nq = cols >> 2;
    const long q = linear_block() * 64 + lane;
    const bool on = q < nq;
    float4* d = reinterpret_cast<float4*>(data);
    float4 a0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), a1 = a0;
    if (on) {
#pragma unroll 4
        for (long r = w; r < rows; r += 32) {
            const float4 x = d[r * nq + q];
            a0.x = __fadd_rn(a0.x, x.x);
            a0.y = __fadd_rn(a0.y, x.y);
            a0.z = __fadd_rn(a0.z, x.z);
            a0.w = __fadd_rn(a0.w, x.w);
            if (r + 16 < rows) {
                const float4 y = d[(r + 16) * nq + q];
                a1.x = __fadd_rn(a1.x, y.x);
                a1.y = __fadd_rn(a1.y, y.y);
                a1.z = __fadd_rn(a1.z, y.z);
                a1.w = __fadd_rn(a1.w, y.w);
            }
        }
    }
    part[w][lane] = make_float4(__fadd_rn(a0.x, a1.x), __fadd_rn(a0.y, a1.y), __fadd_rn(a0.z, a1.z),
                                __fadd_rn(a0.w, a1.w));
    __syncthreads();
    if (w < 4) {   // wave k finishes component k of every lane's 4 columns
        float p[16];
#pragma unroll
        for (int y = 0; y < 16; ++y) {
            const float4 v = part[y][lane];
            p[y] = w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w;
        }
        const float sv = norm_offset(p, rows, factor);
        float* o = reinterpret_cast<float*>(&offs[lane]);
        o[w] = sv;
    }
    __syncthreads();
    if (!on) return;
    const float4 s = offs[lane];
    for (long r = w; r < rows; r += 16) {
        float4 x = d[r * nq + q];
        x.x = __fsub_rn(x.x, s.x);
        x.y = __fsub_rn(x.y, s.y);
        x.z = __fsub_rn(x.z, s.z);
        x.w = __fsub_rn(x.w, s.w);
        d[r * nq + q] = x;
    }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4u __attribute__((aligned(4)));   // rows start at any float

// Float planes of at most 32 NR rows: 4 LANES columns per workgroup, LANES lanes
// of 4 columns by the 32 row partials.  The strip is read once and waits in
// registers (thread y of a lane's column holds rows y, y + 32, ..., which is
// partial y's order) until its columns' offsets are known, then is written.
constexpr int kStripMaxRows = 1536;
template <int NR, int LANES>
__global__ __launch_bounds__(32 * LANES) void normalize_strip_f32_kernel(float* data, long rows, long cols,
                                                                         float factor)
{
    constexpr int kStripCols = 4 * LANES;
    __shared__ f32x4 part[32][LANES];
    __shared__ __align__(16) float offs[kStripCols];
    const int q = threadIdx.x & (LANES - 1), y = threadIdx.x / LANES;
    const long c0 = linear_block() * kStripCols, c = c0 + 4 * q;
    const bool whole = c0 + kStripCols <= cols;   // the strip's, for all threads
    float* col = data + y * cols + c;
    const int mine = rows > y ? (int)((rows - y + 31) / 32) : 0;
    const int left = c < cols ? (int)(cols - c < 4 ? cols - c : 4) : 0;   // columns of this thread
    const int all = (int)(rows / 32);   // rows that every thread has
    f32x4 v[NR];
    f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
    if (whole) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (k < all) v[k] = *reinterpret_cast<const f32x4u*>(col + 32 * k * cols);
            else if (k < mine) v[k] = *reinterpret_cast<const f32x4u*>(col + 32 * k * cols);
        }
    } else {
#pragma unroll
        for (int k = 0; k < NR; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[k][j] = k < mine && j < left ? col[32 * k * cols + j] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < NR; ++k)
        if (k < mine) {
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = __fadd_rn(a[j], v[k][j]);
        }
    part[y][q] = a;
    __syncthreads();
    if (threadIdx.x < kStripCols) {
        const float* f = reinterpret_cast<const float*>(&part[0][0]) + threadIdx.x;
        float p[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = __fadd_rn(f[i * kStripCols], f[(i + 16) * kStripCols]);
        offs[threadIdx.x] = norm_offset(p, rows, factor);
    }
    __syncthreads();
    const f32x4 s = *reinterpret_cast<const f32x4*>(offs + 4 * q);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        f32x4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = __fsub_rn(v[k][j], s[j]);
        if (whole) {
            if (k < mine) *reinterpret_cast<f32x4u*>(col + 32 * k * cols) = x;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k < mine && j < left) col[32 * k * cols + j] = x[j];
        }
    }
}

__global__ void norm_zero_kernel(uint32_t* p, long n)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4u __attribute__((aligned(4)));

// The bytes of 32 consecutive rows, 16 to a lane, from the `blocks` whole ones
// of a segment's 32-row blocks and the `tail` bytes (maybe none) of its last
// rows that start at the lane's.
struct lane_rows {
    int blocks;
    long tail;
};
__device__ __forceinline__ lane_rows rows_of_lane(long i, long r0, long r1, long cols)
{
    return lane_rows{(int)((r1 - r0) / 32), ((r1 - r0) % 32) * cols - 16 * i};
}

// The last 1 to 15 bytes of a lane, zero past them; all loads go out together
// (a loop of loads took 5 us of a 30 us call of one row).
__device__ __forceinline__ u32x4 tail_bytes(const uint8_t* d, int tail)
{
    uint32_t v[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) v[b] = d[b < tail ? b : tail - 1];
    u32x4 x = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 0; b < 16; ++b) x[b >> 2] |= b < tail ? v[b] << (8 * (b & 3)) : 0u;
    return x;
}

// Integer partial sums of one row segment of u8 data: lanes numbered through
// the bytes of 32 consecutive rows, 16 bytes each (32 rows are a whole number
// of them at any column count; a lane's bytes may cross rows), so that every
// lane is busy and byte b of lane i belongs to sum 16 i + b of the 32 x cols
// partials.  Two columns share a 32-bit sum: seg_rows is a multiple of 32 and
// at most kSegRows, whose 256 blocks of 255 fit 16 bits.
constexpr long kSegRows = 32 * 256;
__global__ __launch_bounds__(256) void norm_partial_u8_kernel(const uint8_t* data, long rows, long cols,
                                                              long seg_rows, uint32_t* partial)
{
    __shared__ uint32_t sums[16][257];   // [byte of the lane][lane]
    const long i0 = (long)blockIdx.x * 256, i = i0 + threadIdx.x;
    const long r0 = (long)blockIdx.y * seg_rows;
    const long r1 = rows < r0 + seg_rows ? rows : r0 + seg_rows;
    if (16 * i0 >= (r1 - r0) * cols) return;   // whole work-group: fewer than 32 rows, none of them its
    uint32_t even[4] = {0u, 0u, 0u, 0u}, odd[4] = {0u, 0u, 0u, 0u};
    auto add = [&](u32x4 x) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            even[b] += x[b] & 0x00ff00ffu;
            odd[b] += (x[b] >> 8) & 0x00ff00ffu;
        }
    };
    if (i < 2 * cols) {
        const lane_rows n = rows_of_lane(i, r0, r1, cols);
        const uint8_t* d = data + r0 * cols + 16 * i;
#pragma unroll 8
        for (int k = 0; k < n.blocks; ++k) add(*reinterpret_cast<const u32x4u*>(d + (long)k * 32 * cols));
        d += (long)n.blocks * 32 * cols;
        if (n.tail >= 16) {
            add(*reinterpret_cast<const u32x4u*>(d));
        } else if (n.tail > 0) {
            add(tail_bytes(d, (int)n.tail));
        }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        sums[4 * b][threadIdx.x] = even[b] & 0xffffu;
        sums[4 * b + 1][threadIdx.x] = odd[b] & 0xffffu;
        sums[4 * b + 2][threadIdx.x] = even[b] >> 16;
        sums[4 * b + 3][threadIdx.x] = odd[b] >> 16;
    }
    __syncthreads();
    const long left = 32 * cols - 16 * i0;   // sums from this workgroup's first on
#pragma unroll 4
    for (int k = threadIdx.x; k < 16 * 256; k += 256) {   // a wave adds to 64 neighbouring sums at a time
        const uint32_t a = sums[k & 15][k >> 4];
        if (k < left && a) atomicAdd(partial + 16 * i0 + k, a);
    }
}

// Same, one column per lane, wave w = partials w and w + 16 (u16, and u8 at odd
// bytes).  seg_rows is a multiple of 32, so a row's partial index is its global
// row index mod 32.
template <class T>
__global__ __launch_bounds__(1024) void norm_partial_kernel(const T* data, long rows, long cols, long seg_rows,
                                                            uint32_t* partial)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long c = (long)blockIdx.x * 64 + lane;
    if (c >= cols) return;   // no barrier in this kernel
    const long r0 = (long)blockIdx.y * seg_rows;
    const long r1 = rows < r0 + seg_rows ? rows : r0 + seg_rows;
    uint32_t a0 = 0u, a1 = 0u;
#pragma unroll 4
    for (long r = r0 + w; r < r1; r += 32) {
        a0 += data[r * cols + c];
        if (r + 16 < r1) a1 += data[(r + 16) * cols + c];
    }
    if (a0) atomicAdd(&partial[(long)w * cols + c], a0);
    if (a1) atomicAdd(&partial[(long)(w + 16) * cols + c], a1);
}

// Exact integer partials -> float (exact) -> the reference's tree -> s[c].
__global__ void norm_offsets_kernel(const uint32_t* partial, long rows, long cols, float factor, float* offs)
{
    const long c = (long)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    float p[16];
#pragma unroll
    for (int y = 0; y < 16; ++y)
        p[y] = __fadd_rn((float)partial[(long)y * cols + c], (float)partial[(long)(y + 16) * cols + c]);
    offs[c] = norm_offset(p, rows, factor);
}

// Apply: x' = clamp(x - s[c]).  u8 data: lanes numbered through 32 rows as
// above, four blocks in flight, segments of seg_rows (a multiple of 32) over
// blockIdx.y.
__device__ __forceinline__ uint32_t norm_word(uint32_t x, const float4& s, float maxval)
{
    return (uint32_t)norm_value((float)(x & 0xffu), s.x, maxval) |
           (uint32_t)norm_value((float)((x >> 8) & 0xffu), s.y, maxval) << 8 |
           (uint32_t)norm_value((float)((x >> 16) & 0xffu), s.z, maxval) << 16 |
           (uint32_t)norm_value((float)(x >> 24), s.w, maxval) << 24;
}

__global__ __launch_bounds__(256) void norm_apply_u8_kernel(uint8_t* data, long rows, long cols, long seg_rows,
                                                            const float* __restrict__ offs, float maxval)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 2 * cols) return;
    const long r0 = (long)blockIdx.y * seg_rows;
    const long r1 = rows < r0 + seg_rows ? rows : r0 + seg_rows;
    const lane_rows n = rows_of_lane(i, r0, r1, cols);
    if (n.blocks == 0 && n.tail <= 0) return;
    uint8_t* d = data + r0 * cols + 16 * i;
    float s[16];
    long c = 16 * i % cols;
#pragma unroll
    for (int b = 0; b < 16; ++b) {
        s[b] = offs[c];
        c = c + 1 == cols ? 0 : c + 1;
    }
    const float4 s0 = make_float4(s[0], s[1], s[2], s[3]), s1 = make_float4(s[4], s[5], s[6], s[7]);
    const float4 s2 = make_float4(s[8], s[9], s[10], s[11]), s3 = make_float4(s[12], s[13], s[14], s[15]);
    auto apply = [&](u32x4 x) {
        return u32x4{norm_word(x[0], s0, maxval), norm_word(x[1], s1, maxval), norm_word(x[2], s2, maxval),
                     norm_word(x[3], s3, maxval)};
    };
    const long step = 32 * cols;
    int k = 0;
    for (; k + 3 < n.blocks; k += 4, d += 4 * step) {
        u32x4 x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = *reinterpret_cast<const u32x4u*>(d + j * step);
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4u*>(d + j * step) = apply(x[j]);
    }
    for (; k < n.blocks; ++k, d += step)
        *reinterpret_cast<u32x4u*>(d) = apply(*reinterpret_cast<const u32x4u*>(d));
    if (n.tail >= 16) {
        *reinterpret_cast<u32x4u*>(d) = apply(*reinterpret_cast<const u32x4u*>(d));
    } else if (n.tail > 0) {
        const u32x4 x = apply(tail_bytes(d, (int)n.tail));
#pragma unroll
        for (int b = 0; b < 15; ++b)
            if (b < n.tail) d[b] = (uint8_t)(x[b >> 2] >> (8 * (b & 3)));
    }
}

// Same, one column per lane, rows strided over blockIdx.y.
template <class T>
__global__ void norm_apply_kernel(T* data, long rows, long cols, const float* __restrict__ offs, float maxval)
{
    const long c = (long)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    const float s = offs[c];
    for (long r = blockIdx.y; r < rows; r += gridDim.y)
        data[r * cols + c] = (T)(uint32_t)norm_value((float)data[r * cols + c], s, maxval);
}

inline unsigned blocks_of(long n, long b) { return (unsigned)((n + b - 1) / b); }

template <class T>
hipError_t normalize_int(T* data, long rows, long cols, float factor, int nbits, void* scratch, hipStream_t s)
{
    if (!data || rows < 0 || cols <= 0 || nbits < 1 || nbits > 16) return hipErrorInvalidValue;
    if (rows == 0) return hipSuccess;
    const float maxval = (float)((1u << nbits) - 1u);
    const long type_max = std::is_same<T, uint8_t>::value ? 255 : 65535;
    const bool exact_int = scratch && ((rows + 31) / 32) * type_max <= (1L << 24);
    if (!exact_int) {
        hipLaunchKernelGGL(normalize_columns_kernel<T>, dim3(blocks_of(cols, 64)), dim3(1024), 0, s, data, rows,
                           cols, factor, maxval);
        return hipGetLastError();
    }
    uint32_t* partial = static_cast<uint32_t*>(scratch);
    float* offs = reinterpret_cast<float*>(partial + 32 * cols);
    hipLaunchKernelGGL(norm_zero_kernel, dim3(blocks_of(32 * cols, 256)), dim3(256), 0, s, partial, 32 * cols);
    const bool words = std::is_same<T, uint8_t>::value && (uintptr_t)data % 4 == 0;
    const long colblocks = blocks_of(cols, 64);
    // Row segments (multiples of 32 rows): about 4096 waves, but at least 64
    // rows per lane before it adds its 16 sums to memory (atomics from every
    // XCD are the slow part: with 16 rows per lane 262,144 x 4096 took 930
    // us, x 384 375 us), and at most what 16 bits hold.  Up to 16 segments 16
    // rows are enough: a short chunk waits for its loads, not for the atomics.
    // One column per lane: about 2048 workgroups of 16 waves.
    const long lanes = 2 * cols;
    long nseg = words ? (256 * 1024 + lanes - 1) / lanes : (2048 + colblocks - 1) / colblocks;
    const long short_seg = (rows + 511) / 512, long_seg = (rows + 2047) / 2048;
    const long max_seg = words ? std::max(long_seg, std::min(16L, short_seg)) : short_seg;
    const long min_seg = words ? (rows + kSegRows - 1) / kSegRows : 1;
    if (nseg > max_seg) nseg = max_seg;
    if (nseg < min_seg) nseg = min_seg;
    long seg_rows = (rows + nseg - 1) / nseg;
    seg_rows = (seg_rows + 31) / 32 * 32;
    nseg = (rows + seg_rows - 1) / seg_rows;
    if (words)
        hipLaunchKernelGGL(norm_partial_u8_kernel, dim3(blocks_of(lanes, 256), (unsigned)nseg), dim3(256), 0, s,
                           (const uint8_t*)data, rows, cols, seg_rows, partial);
    else
        hipLaunchKernelGGL(norm_partial_kernel<T>, dim3((unsigned)colblocks, (unsigned)nseg), dim3(1024), 0, s,
                           (const T*)data, rows, cols, seg_rows, partial);
    hipLaunchKernelGGL(norm_offsets_kernel, dim3(blocks_of(cols, 256)), dim3(256), 0, s, (const uint32_t*)partial,
                       rows, cols, factor, offs);
    const unsigned ry = (unsigned)(rows < 2048 ? rows : 2048);
    // 16 rows per lane, 4 where that leaves most of the chip idle (exact_int
    // holds the row count below 65535 segments).
    const long apply_rows = lanes * (rows / 512) < 64 * 1024 ? 128 : 512;
    if (words)
        hipLaunchKernelGGL(norm_apply_u8_kernel,
                           dim3(blocks_of(lanes, 256), (unsigned)((rows + apply_rows - 1) / apply_rows)), dim3(256),
                           0, s, (uint8_t*)data, rows, cols, apply_rows, (const float*)offs, maxval);
    else
        hipLaunchKernelGGL(norm_apply_kernel<T>, dim3(blocks_of(cols, 256), ry), dim3(256), 0, s, data, rows, cols,
                           (const float*)offs, maxval);
    return hipGetLastError();
}

template <int LANES>
hipError_t launch_strips(float* data, long rows, long cols, float factor, hipStream_t s)
{
    const dim3 strips = linear_grid((cols + 4 * LANES - 1) / (4 * LANES), 32 * LANES), threads(32 * LANES);
    if (rows <= 128)
        hipLaunchKernelGGL((normalize_strip_f32_kernel<4, LANES>), strips, threads, 0, s, data, rows, cols, factor);
    else if (rows <= 256)
        hipLaunchKernelGGL((normalize_strip_f32_kernel<8, LANES>), strips, threads, 0, s, data, rows, cols, factor);
    else if (rows <= 512)
        hipLaunchKernelGGL((normalize_strip_f32_kernel<16, LANES>), strips, threads, 0, s, data, rows, cols, factor);
    else if (rows <= 1024)
        hipLaunchKernelGGL((normalize_strip_f32_kernel<32, LANES>), strips, threads, 0, s, data, rows, cols, factor);
    else
        hipLaunchKernelGGL((normalize_strip_f32_kernel<kStripMaxRows / 32, LANES>), strips, threads, 0, s, data, rows,
                           cols, factor);
    return hipGetLastError();
}

}  // namespace

size_t normalize_columns_scratch_bytes(long cols) { return (size_t)(cols > 0 ? cols : 0) * 33u * sizeof(float); }

hipError_t launch_normalize_columns_u8(uint8_t* data, long rows, long cols, float factor, int nbits, void* scratch,
                                       hipStream_t s)
{
    if (nbits > 8) return hipErrorInvalidValue;
    return normalize_int<uint8_t>(data, rows, cols, factor, nbits, scratch, s);
}

hipError_t launch_normalize_columns_u16(uint16_t* data, long rows, long cols, float factor, int nbits,
                                        void* scratch, hipStream_t s)
{
    return normalize_int<uint16_t>(data, rows, cols, factor, nbits, scratch, s);
}

hipError_t launch_normalize_columns_f32(float* data, long rows, long cols, float factor, hipStream_t s)
{
    if (!data || rows < 0 || cols <= 0) return hipErrorInvalidValue;
    if (rows == 0) return hipSuccess;
    // Strips of 64 columns, or of 16 where those would be fewer than 64: 1152 x
    // 3117 floats 34 us with 49 strips and 20 with 195, 1536 x 3000 46 and 20;
    // above, the longer row segments win (512 x 8000 7.4 us against 16.8).
    // Of up to 4 rows most of a strip's threads have none: 1 x 500,000 9.9 us by
    // columns of 4 against 11.2, 4 x 500,000 11.0 against 11.9; 6 rows 12.8
    // against 12.4.
    const bool columns4 = cols % 4 == 0 && (uintptr_t)data % 16 == 0 && cols >= 160 * 256;
    if (rows <= kStripMaxRows && !(rows <= 4 && columns4))
        return cols >= 64 * 64 ? launch_strips<16>(data, rows, cols, factor, s)
                               : launch_strips<4>(data, rows, cols, factor, s);
    // Taller planes are read twice, 4 columns per lane where that leaves enough
    // workgroups of 256 columns: 1600 x 50,000 177 us against 218 with one column
    // per lane, 6080 x 111,328 1.68 ms against 1.86; 3072 x 32,768 256 us against
    // 244, 1600 x 20,000 65 against 62.
    if (columns4)
        hipLaunchKernelGGL(normalize_columns_f32x4_kernel, linear_grid((cols / 4 + 63) / 64, 1024), dim3(1024), 0, s,
                           data, rows, cols, factor);
    else
        hipLaunchKernelGGL(normalize_columns_kernel<float>, linear_grid((cols + 63) / 64, 1024), dim3(1024), 0, s, data,
                           rows, cols, factor, 0.0f);
    return hipGetLastError();
}

}  // namespace aa_hip

// Dedispersion of u8 rows on the matrix cores, for gfx950.
//
// For a tile of 16 DM trials and a group of neighbouring channels, choose a
// base delay base(d) per trial (the delay of the group's middle channel) and a
// byte offset off(c) per channel, so that
//     delay(c, d) = base(d) + off(c) + r(c, d),   0 <= r(c, d) < 4 (or 8, 16).
// The group's part of out[d][t] is then P[d][t + base(d)] with
//     P[d][k] = sum_c sum_{x < 4} S[d][c, x] L[c][k + off(c) + x],
// S one-hot in x (x = r(c, d)): a product of the 0/1 matrix S (16 trials x
// 16 channels x 4 bytes = 64) with the rows, which is one
// v_mfma_i32_16x16x64_i8 per 16 samples and 16 channels.  Every sum is an
// exact integer, so the result is the reference's whatever the grouping.
//
// "Slots" generalise the channels: a slot is 4 consecutive byte positions of
// one channel; a channel whose r spans up to 4 n values takes n slots.  A step
// is 16 slots (K = 64).  A slot is narrow if its selectors use 3 of its 4
// positions: an odd sample can then take its even neighbour's operand and the
// selectors a byte higher, which saves half of the operand alignments.  The
// host plans groups, slots and selectors once per range (matrix_plan), widths
// as even as they can be and the narrow slots of a group first; 74 to 90 % of
// the steps of the plans below are narrow.
//
// Work-group: 8 waves, 16 DM trials, a window of 8 x 240 positions k.  Per step
// a wave loads, for each of its lane's 4 slots, the 16 bytes at its own
// positions (lane m of 16 holds positions 16 m .. 16 m + 15 of the wave's run)
// and builds the operand of positions 16 m + q with v_alignbyte, q = 0..15:
// 16 products per step, accumulated over the steps of the group.  The loads
// are of whole dwords (loads at odd bytes run at 16 B per clock and CU, a
// quarter of whole dwords); the bytes left over are shifted out in registers.
// The last lane of 16 only feeds its neighbour, hence 240 and not 256: loading
// its missing dword instead cost 45 ms of 190 on the 8-range plan.  Bytes are
// flipped to signed (x ^ 0x80) for the signed product; the sums of the 128s
// taken off are added back at the end.
//
// At the end of a group the waves write P as 16-bit values to LDS, one row per
// trial, and after one barrier wave w adds trials 2 w and 2 w + 1 at their own
// base delays to 32-bit sums.  Rows of trials with an odd base delay are
// written one sample to the left: reading dwords at odd samples cost 26 ms of
// 190.  The step records (selectors, slot addresses) go through LDS, one wave
// loading each, and what steers the loop is read with scalar loads: a vector
// load for it waits for the row loads before it.
//
// Bound: vector instruction issue and the hand-over of the groups.  A step is
// 60 vector instructions if narrow (32 alignments, 16 sign flips, 8 lane
// moves, 4 selectors), 88 if not, beside 16 products per wave; issue takes 4.3
// cycles per instruction and about half of a product's 16 does not overlap
// with it.  With all alignments and flips left out the 8-range plan would take
// 76 ms; LDS is 13 % busy, the vector memory return path about two thirds.
// Tried and not kept: three row buffers (no change), the sums of a group
// delayed into the next group's first step (99.9 against 99.2 ms), a fixed
// interleave of products and vector instructions (99.2 against 97.6 ms).
//
// Measured on the 8-range plan (4096 channels x 1,048,576 samples, 6080
// trials, 1.48e13 channel-adds): 85 ms for the 8 launches, 174 T adds/s,
// against 238.6 ms with the pair shapes and 92.7 ms with wide steps only; the
// single-range plan (512 channels x 131,072 samples, 1024 trials) 0.75 ms
// against 1.19 and 0.79.
#include "ddtr_matrix.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace aa_hip {

namespace {

constexpr int kMatDms = 16;
constexpr int kMatWaves = 8;
constexpr int kMatThreads = 64 * kMatWaves;
constexpr int kMatRun = 240;                     // window positions per wave (15 lanes of 16)
constexpr int kMatWin = kMatRun * kMatWaves;     // window positions per tile
constexpr int kMatRow = kMatWin / 2 + 4;         // dwords per LDS row (rows 4 banks apart modulo 32)
constexpr int kMatOut = kMatWin / 128;           // dwords per lane of a trial's tile
constexpr int kMatGroupMax = 256;                // channels: 16-bit partial sums
constexpr int kMatMinOut = 1024;                 // smallest tile worth its window

typedef uint32_t u32x4m __attribute__((ext_vector_type(4)));
typedef u32x4m u32x4a __attribute__((aligned(4)));   // 16 bytes at a whole dword
typedef int i32x4 __attribute__((ext_vector_type(4)));

struct mat_tile {
    int group0, ngroups;   // groups of this DM tile
    int step0, nsteps;     // their steps
};
struct mat_group {
    int nsteps, narrow;    // steps, the first ones narrow
    int odd;               // bit d: trial d's first sample is the odd one of its dword
    int shift;             // the sums' weight: 8 for a group of high bytes
    int e[kMatDms];        // dword of each trial's first sample in its LDS row
};
struct mat_step {
    uint32_t sel[64][4];   // [lane][slot of the lane]: selector dwords
    uint32_t off[16];      // slot addresses (whole dwords) from base
    uint32_t shift[16];    // and the bytes left over
    long long base;        // byte address (from the level) of the step's lowest slot
    long long pad;
};

// Tables read with scalar loads: in the vector memory queue they would wait
// for the row loads issued before them.
typedef __attribute__((address_space(4))) mat_group const_group;
typedef __attribute__((address_space(4))) mat_step const_step;

struct mat_args {
    lds_params p;
    const mat_tile* tiles;
    const mat_group* groups;
    const mat_step* steps;
    int tile_out;
    const int* over;       // 64 entries: more than half of them set: flag every tile
    int* flags;
    int t_flags;           // samples that can set a tile's flag
};

__shared__ uint32_t m_rows[2 * kMatDms * kMatRow + 512];   // the tail: reads past the last row's window
// The records of two chunks of kMatWaves steps: every wave reads all of them.
struct mat_meta {
    u32x4m sel[64];
    u32x4m off[4], shift[4];
};
__shared__ mat_meta m_meta[2][kMatWaves];

struct mat_raw {
    u32x4m q[4];           // 16 bytes of each slot, from a whole dword on
    u32x4m shift;          // bytes from there to the slot's first position
    u32x4m sel;
};

// One step's 16 products.  Lane m of 16 holds bytes 16 m .. 16 m + 15 of its 4
// slots; the dwords after them are the next lane's first ones (lane 15 has
// none: its positions from 8 on are not used).
// NARROW: no slot's selectors use the last of its 4 positions, so that a pair of
// positions 16 m + q, q even, shares an operand: the odd one takes the
// selectors a byte higher.
template <bool FIRST, bool NARROW>
__device__ __forceinline__ void mat_step_products(const mat_raw& r, i32x4 (&acc)[16])
{
    asm volatile("; products %0 %1" ::"n"((int)FIRST), "n"((int)NARROW));   // keeps the copies apart
    uint32_t D[4][5];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t R[5];
#pragma unroll
        for (int k = 0; k < 4; ++k) R[k] = r.q[j][k] ^ 0x80808080u;
        R[4] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)R[0], 0x101, 0xf, 0xf, true);   // row_shl:1
#pragma unroll
        for (int k = 0; k < 4; ++k) D[j][k] = __builtin_amdgcn_alignbyte(R[k + 1], R[k], r.shift[j]);
        D[j][4] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)D[j][0], 0x101, 0xf, 0xf, true);   // row_shl:1
    }
    i32x4 b[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        b[0][j] = (int)r.sel[j];
        b[1][j] = (int)(r.sel[j] << 8);
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int sh = NARROW ? q & 2 : q & 3;
        i32x4 a;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            a[j] = sh ? (int)__builtin_amdgcn_alignbyte(D[j][q / 4 + 1], D[j][q / 4], sh) : (int)D[j][q / 4];
        const i32x4 zero = {0, 0, 0, 0};
        acc[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b[NARROW ? q & 1 : 0], FIRST ? zero : acc[q], 0, 0, 0);
    }
}

// PLANES: 16-bit samples as planes of low and high bytes.
template <bool PLANES>
__global__ __launch_bounds__(kMatThreads, 2) void dedisperse_matrix_kernel(mat_args a)
{
    const lds_params& p = a.p;
    const int ntiles = p.n_dm_tiles * p.n_t_tiles;
    // work-group g runs on XCD g % 8: each XCD takes a run of consecutive
    // tiles, DM tiles of one time tile after another, which share their rows
    const int per = (ntiles + 7) / 8;
    const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || tile >= ntiles) return;   // whole work-group, before any barrier
    const int t_tile = tile / p.n_dm_tiles, dm_tile = tile - t_tile * p.n_dm_tiles;
    if (PLANES && __popcll(__ballot(a.over[threadIdx.x & 63] != 0)) > 32) {
        if (threadIdx.x == 0) a.flags[tile] = 1;
        return;   // whole work-group, before any barrier
    }
    const long t0 = (long)t_tile * a.tile_out;
    const mat_tile tl = a.tiles[dm_tile];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int m = lane & 15, kb = lane >> 4;
    const uint32_t vlane = (uint32_t)(wave * kMatRun + m * 16);
    const uint8_t* __restrict__ L = p.L + t0;
    const mat_step* __restrict__ steps = a.steps + tl.step0;
    const const_step* csteps = (const const_step*)(uintptr_t)steps;
    const const_group* groups = (const const_group*)(uintptr_t)(a.groups + tl.group0);
    const int S = tl.nsteps;

    i32x4 acc[16];
    int lo[2][kMatOut], hi[2][kMatOut];
#pragma unroll
    for (int dd = 0; dd < 2; ++dd)
#pragma unroll
        for (int j = 0; j < kMatOut; ++j) lo[dd][j] = hi[dd][j] = 0;
    // Step records come in chunks of 8: wave w loads record w of a chunk, a
    // chunk ahead of its use, and hands it to the other waves through LDS.
    u32x4m rec_sel, rec_off;
    auto load_rec = [&](int chunk) {
        const int i = chunk * kMatWaves + wave;
        const mat_step& st = steps[i < S ? i : S - 1];
        rec_sel = *reinterpret_cast<const u32x4m*>(st.sel[lane]);
        rec_off = *reinterpret_cast<const u32x4m*>(st.off + 4 * (lane & 7));   // off[16], shift[16]
    };
    auto keep_rec = [&](int chunk) {
        mat_meta& m = m_meta[chunk & 1][wave];
        m.sel[lane] = rec_sel;
        if (lane < 8) m.off[lane] = rec_off;
    };
    int f = 0;   // the next step to fetch; its addresses are at hand
    long long base = csteps[0].base;
    u32x4m off;
    auto meta_of = [&](int i) -> const mat_meta& { return m_meta[(i / kMatWaves) & 1][i & (kMatWaves - 1)]; };
    auto fetch = [&](mat_raw& r) {
        const uint8_t* b = L + base;
        base = csteps[f + 1 < S ? f + 1 : S - 1].base;
#pragma unroll
        for (int j = 0; j < 4; ++j) r.q[j] = *reinterpret_cast<const u32x4a*>(b + (size_t)(off[j] + vlane));
        const mat_meta& m = meta_of(f);
        r.sel = m.sel[lane];
        r.shift = m.shift[kb];
        ++f;
        if ((f & (kMatWaves - 1)) == 0) {   // a new chunk of records: the one before it has been read
            __syncthreads();
            keep_rec(f / kMatWaves + 1);
            load_rec(f / kMatWaves + 2);
        }
        off = meta_of(f).off[kb];
    };

    load_rec(0);
    keep_rec(0);
    load_rec(1);
    __syncthreads();
    keep_rec(1);
    load_rec(2);
    off = meta_of(0).off[kb];
    mat_raw A, B;
    fetch(A);
    int s = 0, g = 0, left = groups[0].nsteps, narrow = groups[0].narrow;
    bool first = true;

    auto body = [&](mat_raw& cur, mat_raw& fill) {
        fetch(fill);
        if (narrow > 0) {
            if (first) mat_step_products<true, true>(cur, acc);
            else mat_step_products<false, true>(cur, acc);
        } else {
            if (first) mat_step_products<true, false>(cur, acc);
            else mat_step_products<false, false>(cur, acc);
        }
        --narrow;
        first = false;
        ++s;
        if (--left == 0) {
            // The group's P: the lane holds trial m at positions 16 (4 kb + i)
            // + q.  A row starts at the trial's first sample rounded down to
            // two (trials with an odd base are written one sample to the
            // left), so that the sums read whole dwords.
            const const_group& gr = groups[g];
            uint32_t* rows = m_rows + (g & 1) * (kMatDms * kMatRow);
            uint32_t* w = rows + m * kMatRow + wave * (kMatRun / 2) + kb * 32;
            const uint32_t odd = ((uint32_t)gr.odd >> m & 1u) * 16u;
            const uint32_t next = (uint32_t)__shfl(acc[0][0], (lane + 16) & 63);   // the run after the lane's last
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t k[9];
#pragma unroll
                for (int h = 0; h < 8; ++h)
                    k[h] = __builtin_amdgcn_perm((uint32_t)acc[2 * h + 1][i], (uint32_t)acc[2 * h][i], 0x05040100u);
                k[8] = i < 3 ? (uint32_t)acc[0][i < 3 ? i + 1 : 3] : kb < 3 ? next : 0u;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4m v;
#pragma unroll
                    for (int n = 0; n < 4; ++n) v[n] = __builtin_amdgcn_alignbit(k[4 * h + n + 1], k[4 * h + n], odd);
                    if (i < 3 || kb < 3) *reinterpret_cast<u32x4m*>(w + 8 * i + 4 * h) = v;
                }
            }
            __syncthreads();
#pragma unroll
            for (int dd = 0; dd < 2; ++dd) {
                const uint32_t* row = rows + (2 * wave + dd) * kMatRow + gr.e[2 * wave + dd] + lane;
                if (PLANES && gr.shift) {
#pragma unroll
                    for (int j = 0; j < kMatOut; ++j) {
                        const uint32_t v = row[64 * j];
                        lo[dd][j] += (int)(short)v * 256;
                        hi[dd][j] += ((int)v >> 16) * 256;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < kMatOut; ++j) {
                        const uint32_t v = row[64 * j];
                        lo[dd][j] += (int)(short)v;
                        hi[dd][j] += (int)v >> 16;
                    }
                }
            }
            ++g;
            left = s < S ? groups[g].nsteps : 0;
            narrow = s < S ? groups[g].narrow : 0;
            first = true;
        }
    };
    for (;;) {
        body(A, B);
        if (s >= S) break;
        body(B, A);
        if (s >= S) break;
    }

    const long t_end = t0 + a.tile_out < p.t_processed ? t0 + a.tile_out : (long)p.t_processed;
    const int bias = 128 * p.nchans * (PLANES ? 257 : 1);   // what the sign flips took off every sum
    // A sum whose float adds round.  Looked for in all samples that the rows hold,
    // also those past t_processed: calls of different lengths that overlap on
    // other streams then write the same flags.
    const long f_end = PLANES ? (t0 + a.tile_out < a.t_flags ? t0 + a.tile_out : (long)a.t_flags) : 0;
    bool above = false;
#pragma unroll
    for (int dd = 0; dd < 2; ++dd) {
        const int d = dm_tile * kMatDms + 2 * wave + dd;
        if (d >= p.ndms) continue;
        float* orow = p.out + (size_t)d * p.out_pitch;
        const bool aligned = ((uintptr_t)orow & 7) == 0;
#pragma unroll
        for (int j = 0; j < kMatOut; ++j) {
            const long t = t0 + 2 * (lane + 64 * j);
            const uint32_t s0 = (uint32_t)(lo[dd][j] + bias), s1 = (uint32_t)(hi[dd][j] + bias);
            if (PLANES) above |= (t < f_end && s0 > (1u << 24)) || (t + 1 < f_end && s1 > (1u << 24));
            const float v0 = out_value(s0, p), v1 = out_value(s1, p);
            if (aligned && t + 1 < t_end) {
                *reinterpret_cast<float2*>(orow + t) = make_float2(v0, v1);
            } else {
                if (t < t_end) orow[t] = v0;
                if (t + 1 < t_end) orow[t + 1] = v1;
            }
        }
    }
    if (PLANES) {
        const int any = __syncthreads_or(above);
        if (threadIdx.x == 0) a.flags[tile] = any ? 1 : 0;
    }
}

// ------------------------------------------------------------------ planning

// Span of delay(c, d) - delay(ref, d) over the tile's trials, in 16 bits
// (differences inside a group are far smaller; emission checks in 32 bits).
inline void rel_span(const int16_t* row, const int16_t* ref, int& lo, int& hi)
{
    int16_t a = 32767, b = -32768;
    for (int d = 0; d < kMatDms; ++d) {
        const int16_t v = (int16_t)(row[d] - ref[d]);
        a = std::min(a, v);
        b = std::max(b, v);
    }
    lo = a;
    hi = b;
}

struct tile_delays {
    const int* d32;        // [c][16]
    const int16_t* d16;
    int nchans;
};

// Slots of a channel whose r spans `span` values, as even as they can be: of
// them, wide ones (4 values; the others 3 or fewer).
inline int slots_of(int span) { return (span + 3) / 4; }
inline int wide_of(int span) { return std::max(0, span - 3 * slots_of(span)); }

// Whether channels [c0, c0 + n) with reference channel `ref` span at most
// `limit` values each, at non-negative row offsets.
bool group_fits(const tile_delays& t, int c0, int n, int ref, int limit, int* slots, int* wide)
{
    const int16_t* r16 = t.d16 + (size_t)ref * kMatDms;
    const int* r32 = t.d32 + (size_t)ref * kMatDms;
    int w0 = r32[0];
    for (int d = 1; d < kMatDms; ++d) w0 = std::min(w0, r32[d]);
    int total = 0, w = 0;
    for (int c = c0; c < c0 + n; ++c) {
        int lo, hi;
        rel_span(t.d16 + (size_t)c * kMatDms, r16, lo, hi);
        const int span = hi - lo + 1;
        if (span > limit || w0 + lo < 0) return false;
        total += slots_of(span);
        w += wide_of(span);
    }
    *slots = total;
    *wide = w;
    return true;
}

// Work of a plan in units of one step with wide slots (about 1600 cycles per
// work-group); the hand-over of a group through LDS takes about 2000 cycles.
constexpr double kNarrowCost = 0.8;
constexpr double kGroupCost = 1.2;

struct group_pick {
    int n = 0, ref = 0, slots = 0, wide = 0;
    int steps() const { return (slots + 15) / 16; }
    int narrow_steps() const { return wide ? (slots - wide) / 16 : steps(); }   // the steps without a wide slot
    double cost() const { return steps() - (1.0 - kNarrowCost) * narrow_steps() + kGroupCost; }
};

group_pick fit(const tile_delays& t, int c0, int n, int limit)
{
    group_pick g;
    int slots = 0, wide = 0;
    for (int ref : {c0 + n / 2, c0})   // the first channel where the middle one would read before the rows
        if (group_fits(t, c0, n, ref, limit, &slots, &wide)) {
            g = group_pick{n, ref, slots, wide};
            break;
        }
    return g;
}

// The largest group from c0 (trimmed to whole steps where it spans several).
group_pick pick_group(const tile_delays& t, int c0, int limit, int guess)
{
    const int room = std::min(t.nchans - c0, kMatGroupMax);
    int good = 0, bad = room + 1, n = std::max(1, std::min(guess, room));
    group_pick best;
    for (int stride = std::max(1, n / 4); bad - good > 1;) {
        const group_pick g = fit(t, c0, n, limit);
        if (g.n) {
            best = g;
            good = n;
        } else {
            bad = n;
        }
        if (bad == room + 1) {
            n = std::min(room, good + stride);
            stride *= 2;
        } else if (good == 0) {
            n = std::max(1, bad - stride);
            stride *= 2;
        } else {
            n = (good + bad) / 2;
        }
    }
    if (best.n == 0 || best.n == t.nchans - c0) return best;
    for (int cut = 1; cut < 16 && best.slots > 16 && best.slots % 16; ++cut) {
        const group_pick g = fit(t, c0, good - cut, limit);
        if (!g.n || g.slots <= 16) break;
        if (g.slots % 16 == 0) return g;
    }
    return best;
}

// Cost of the pair shapes in the same units: 16 channels of one of their
// tiles, which shorten with the trials' spread.  Break-even measured on plans
// of 128 to 4096 channels: at 3.2 (144 channels, 0.120 ms both ways) and at
// 3.9 (165 channels) this kernel is level or ahead (0.85 against 0.93 ms), at
// 5.1 (155 channels) behind (1.43 against 1.34 ms).
double pair_cost(int nchans, int spread)
{
    const double tile = spread <= 268 ? 2016.0 : spread <= 520 ? 1512.0 : 1008.0;
    return 4.2 * nchans / 16.0 / tile;
}

}  // namespace

matrix_layout matrix_plan(const float* h_dmshifts, int nchans, int ndms, float mstartdm, float mdmstep, size_t pitch,
                          std::vector<uint8_t>* bytes, int planes)
{
    matrix_layout lay;
    if (nchans < 1 || ndms < 1 || (size_t)pitch * 17 >= (1ull << 32) || (planes == 2 && nchans > 65536)) return lay;
    // Against the 16-bit LDS kernel (5.75 T channel-adds/s where the pair
    // shapes do 54) any plan pays that is not 8 times the pair shapes' cost.
    const double limit_cost = planes == 2 ? 8.0 : 1.0;
    const int ntiles = (ndms + kMatDms - 1) / kMatDms;
    std::vector<float> shift((size_t)ntiles * kMatDms);
    for (int d = 0; d < ntiles * kMatDms; ++d)   // trials past the last repeat it
        shift[(size_t)d] = __builtin_fmaf((float)std::min(d, ndms - 1), mdmstep, mstartdm);

    std::vector<int> d32((size_t)nchans * kMatDms);
    std::vector<int16_t> d16((size_t)nchans * kMatDms);
    std::vector<mat_tile> tiles;
    std::vector<mat_group> groups;
    std::vector<mat_step> steps;
    struct pick_list {
        std::vector<group_pick> g;
        long nsteps = 0;
    };
    int spread = 0;
    double cost = 0.0;
    int limit_guess = 4;
    for (int tile = 0; tile < ntiles; ++tile) {
        const float* st = shift.data() + (size_t)tile * kMatDms;
        for (int c = 0; c < nchans; ++c)
            for (int d = 0; d < kMatDms; ++d) {
                const float prod = h_dmshifts[c] * st[d];
                d32[(size_t)c * kMatDms + d] = (int)prod;
                d16[(size_t)c * kMatDms + d] = (int16_t)(int)prod;
            }
        const tile_delays t{d32.data(), d16.data(), nchans};
        pick_list best;
        double best_cost = INFINITY;
        for (int limit : {4, 6, 8, 12, 16}) {
            if (tile > 0 && limit != limit_guess) continue;   // one limit per range: the first tile's best
            pick_list l;
            int guess = 64;
            bool ok = true;
            double w = 0.0;
            for (int c = 0; c < nchans && ok;) {
                const group_pick g = pick_group(t, c, limit, guess);
                ok = g.n > 0;
                if (!ok) break;
                l.g.push_back(g);
                l.nsteps += g.steps();
                w += g.cost();
                guess = g.n;
                c += g.n;
            }
            if (ok && w < best_cost) {
                best_cost = w;
                best = l;
                if (tile == 0) limit_guess = limit;
            }
        }
        if (best.g.empty() || (tile == 0 && best_cost / kMatWin > 1.5 * limit_cost * pair_cost(nchans, 0))) return lay;   // far off
        cost += planes * best_cost;
        mat_tile tl{(int)groups.size(), planes * (int)best.g.size(), (int)steps.size(), planes * (int)best.nsteps};
        for (int plane = 0; plane < planes; ++plane) {
            int c0 = 0;
            for (const group_pick& pk : best.g) {
                mat_group gr{};
                gr.shift = 8 * plane;
                gr.nsteps = pk.steps();
                gr.narrow = pk.narrow_steps();
                const int* base = d32.data() + (size_t)pk.ref * kMatDms;
                const int w0 = *std::min_element(base, base + kMatDms);
                for (int d = 0; d < kMatDms; ++d) {
                    gr.e[d] = (base[d] - w0) / 2;
                    gr.odd |= ((base[d] - w0) & 1) << d;
                    spread = std::max(spread, base[d] - w0);
                }
                int slot = 0;
                long long addr[16];
                bool near = true;   // slots within the kernel's 32-bit offsets
                auto close_step = [&]() {
                    mat_step& ms = steps.back();
                    long long lowest = addr[0];
                    for (int k = 1; k < 16; ++k) lowest = std::min(lowest, addr[k]);
                    ms.base = lowest & ~3ll;
                    for (int k = 0; k < 16; ++k) {
                        const long long off = (addr[k] & ~3ll) - ms.base;
                        near = near && off < (1ll << 32) - 2 * kMatWin;
                        ms.off[k] = (uint32_t)off;
                        ms.shift[k] = (uint32_t)(addr[k] & 3);
                    }
                };
                // narrow slots first, then the wide ones
                struct part {
                    int c, start, width;   // channel, first r (from the channel's lowest delay - base), values
                };
                std::vector<part> narrow, wide;
                for (int c = c0; c < c0 + pk.n; ++c) {
                    const int* row = d32.data() + (size_t)c * kMatDms;
                    int lo = row[0] - base[0], hi = lo;
                    for (int d = 1; d < kMatDms; ++d) {
                        lo = std::min(lo, row[d] - base[d]);
                        hi = std::max(hi, row[d] - base[d]);
                    }
                    const int span = hi - lo + 1;
                    if (span > 16 || w0 + lo < 0) return lay;   // the 16-bit spans disagree
                    for (int k = 0, r = lo; k < slots_of(span); ++k) {
                        const bool w = k < wide_of(span);
                        const int width = std::min(w ? 4 : 3, hi + 1 - r);
                        (w ? wide : narrow).push_back(part{c, r, width});
                        r += width;
                    }
                }
                if ((int)(narrow.size() + wide.size()) != pk.slots || (int)wide.size() != pk.wide) return lay;
                narrow.insert(narrow.end(), wide.begin(), wide.end());
                for (const part& pt : narrow) {
                    const int k = slot & 15;
                    if (k == 0) steps.emplace_back();
                    addr[k] = ((long long)plane * nchans + pt.c) * (long long)pitch + w0 + pt.start;
                    const int* row = d32.data() + (size_t)pt.c * kMatDms;
                    auto& out = steps.back().sel;
                    for (int d = 0; d < kMatDms; ++d) {
                        const int r = row[d] - base[d] - pt.start;
                        // lane (d, slot / 4), dword slot % 4
                        if (r >= 0 && r < pt.width) out[(k >> 2) * 16 + d][k & 3] = 1u << (8 * r);
                    }
                    if (k == 15) close_step();
                    ++slot;
                }
                if (slot & 15) {   // unused slots: any readable address, zero selectors
                    for (int k = slot & 15; k < 16; ++k) addr[k] = addr[(slot & 15) - 1];
                    close_step();
                }
                if (!near) return lay;
                groups.push_back(gr);
                c0 += pk.n;
            }
        }
        tiles.push_back(tl);
    }
    const int tile_out = (kMatWin - spread) / 16 * 16;
    if (tile_out < kMatMinOut) return lay;
    if (cost / ntiles / tile_out > limit_cost * pair_cost(nchans, spread)) return lay;

    auto align = [](size_t v) { return (v + 255) / 256 * 256; };
    lay.n_dm_tiles = ntiles;
    lay.tile_out = tile_out;
    lay.tile_cost = (float)(cost / ntiles);
    lay.planes = planes;
    lay.off_group = align(tiles.size() * sizeof(mat_tile));
    lay.off_step = align(lay.off_group + groups.size() * sizeof(mat_group));
    lay.bytes = lay.off_step + steps.size() * sizeof(mat_step);
    if (bytes) {
        bytes->resize(lay.bytes);
        std::memcpy(bytes->data(), tiles.data(), tiles.size() * sizeof(mat_tile));
        std::memcpy(bytes->data() + lay.off_group, groups.data(), groups.size() * sizeof(mat_group));
        std::memcpy(bytes->data() + lay.off_step, steps.data(), steps.size() * sizeof(mat_step));
    }
    return lay;
}

// Time model in us, fitted on 800 ranges of 8 to 2000 channels, 1 to 1000 trials
// of fine and coarse steps, 200 to 200,000 samples (both kernels with all their
// passes, 12 % standard error each): the matrix kernel's tiles one per CU, 12 us
// to start and end one and 0.86 per step, after the byte planes are made;
// dedisperse_u16's tiles of 512 samples about two per CU, 0.79 us per channel.
// With it no range of those is more than 7 % slower than by the other kernel;
// without, 40 channels x 1000 trials 2 DM units apart x 200,000 samples took 2.38
// ms in place of 1.61, 16 x 64 x 4000 39 us in place of 21.  Below 24 channels the
// matrix kernel gains 5 % at most.
bool matrix_beats_u16(int nchans, long t, const matrix_layout& lay)
{
    if (nchans < kU16MatrixMinChannels || lay.tile_out <= 0 || t <= 0) return false;
    const double tiles = (double)lay.n_dm_tiles * (double)((t + lay.tile_out - 1) / lay.tile_out) / 256.0;
    const double rounds = tiles <= 1.0 ? 1.0 : tiles < 2.0 ? 2.0 : tiles;
    const double matrix = 4.0 + rounds * (12.0 + 0.86 * lay.tile_cost) + 1.75e-6 * nchans * t;
    const double u16_tiles = (double)lay.n_dm_tiles * (double)((t + 511) / 512) / (1.9 * 256.0);
    const double u16 = 8.0 + std::max(1.0, u16_tiles) * 0.79 * nchans + 1.9e-6 * nchans * t;
    return matrix < u16;
}

hipError_t launch_dedisperse_matrix(const lds_params& p, const matrix_layout& lay, hipStream_t s, const int* over,
                                    int* flags, int t_flags)
{
    if (p.ndms <= 0 || p.t_processed <= 0) return hipSuccess;
    if ((lay.planes == 2) != (over && flags) || (flags && t_flags < p.t_processed)) return hipErrorInvalidValue;
    if (!p.pair_recs || lay.tile_out <= 0 || lay.n_dm_tiles != (p.ndms + kMatDms - 1) / kMatDms)
        return hipErrorInvalidValue;
    mat_args a{};
    a.p = p;
    a.p.n_dm_tiles = lay.n_dm_tiles;
    a.p.n_t_tiles = (p.t_processed + lay.tile_out - 1) / lay.tile_out;
    a.tile_out = lay.tile_out;
    a.over = over;
    a.flags = flags;
    a.t_flags = t_flags;
    const char* t = static_cast<const char*>(p.pair_recs);
    a.tiles = reinterpret_cast<const mat_tile*>(t);
    a.groups = reinterpret_cast<const mat_group*>(t + lay.off_group);
    a.steps = reinterpret_cast<const mat_step*>(t + lay.off_step);
    const long tiles = (long)a.p.n_dm_tiles * a.p.n_t_tiles;
    if (tiles > 0x7ffffff0L) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
    if (lay.planes == 2) hipLaunchKernelGGL(dedisperse_matrix_kernel<true>, grid, dim3(kMatThreads), 0, s, a);
    else hipLaunchKernelGGL(dedisperse_matrix_kernel<false>, grid, dim3(kMatThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace aa_hip

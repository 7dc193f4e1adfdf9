// Batched DM refinement of candidate windows (see frac_refine.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace aa_hip {

constexpr int kRefineMaxSamples = 4096;    // per window
constexpr int kRefineMaxChannels = 4096;   // per window
constexpr int kRefineThreads = 256;
constexpr int kRefineSeg = 1024;           // samples of an item
constexpr int kRefineChunk = 256;          // channels of an item at most
constexpr int kRefineChunkMin = 16;        // (a plan's own number: refine_chunk)
constexpr int kRefineScan = 3;             // scan points of a pass

struct refine_cand {
    int64_t x_off;      // window at x + x_off, [C][T] float32
    int64_t ds_off;     // delay per unit DM at ds + ds_off, C entries
    int64_t power_off;  // channel powers at power + power_off, C entries (loss 1)
    int64_t part_off;   // partial profiles at part + part_off
    int C, T;
};

// Part of one window: channels c0 .. c0 + nc - 1 (chunk number c0 / the plan's
// chunk), samples seg * kRefineSeg on.
struct refine_item {
    int cand, chunk, c0, nc, seg;
};

// Partial profiles of one window: a chunk holds up to kRefineScan rows of
// T + (T - 1) / kRefineSeg entries.
inline int64_t refine_part_entries(int C, int T, int chunk)
{
    return (int64_t)((C + chunk - 1) / chunk) * kRefineScan * (T + (T - 1) / kRefineSeg);
}

// Channels per item for a plan's windows: kRefineChunk, halved while the items
// are fewer than four per CU and an item's channels (each lane's serial loop)
// still outweigh the chunks that the combine pass then adds.
int refine_chunk(int ncand, const int* nchans, const int* nsamp);

// A candidate between evaluations.
struct refine_state {
    float u, step, best_u;
    double prev, best_l, pad;
};

struct refine_args {
    const float* x;
    const float* ds;
    const refine_cand* cands;   // [ncand]
    const refine_item* items;   // [nitems], longest first
    int ncand, nitems;
    int chunk;                  // channels of an item
    int longest;                // most samples of a window
    float* u;                   // [ncand] residual DM, updated in place
    float* step;                // [ncand] Rprop step, updated in place
    double* prev_grad;          // [ncand] previous dL/du, updated in place
    double* loss;               // [ncand] L at the final u
    double* grad;               // [ncand] dL/du at the final u
    int nsteps;
    float step_max, step_min;
    int scan_n;                 // coarse scan points before the steps (0 = none)
    float scan_lo, scan_step;   // scan offsets relative to the starting u
    refine_state* cur;          // [ncand]
    double* best_grad;          // [ncand]
    double* scan_loss;          // [ncand][kRefineScan]
    double* part;               // partial profiles
    int loss_kind;              // 0: E = sum_t y^2; 1: E minus the expected noise energy
    double* power;              // loss 1: per-candidate channel powers (written by the launch)
};

hipError_t launch_refine(const refine_args& a, hipStream_t s);

}  // namespace aa_hip

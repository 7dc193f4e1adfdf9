// Dedispersion on the matrix cores (see ddtr_matrix.hip for the algorithm).
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "ddtr_lds.h"

namespace aa_hip {

// Internal number of this kernel beside the LDS chunk shapes 0-6.
constexpr int kShapeMatrix = kLdsVariants;

// Where the parts of a range's plan tables lie, and the tile they are for.
struct matrix_layout {
    int n_dm_tiles = 0;
    int tile_out = 0;      // output samples per tile (0: the range does not take this kernel)
    float tile_cost = 0;   // a tile's work in steps with wide slots
    int planes = 1;        // 2: 16-bit samples as two planes of byte rows, low bytes then high bytes
    size_t off_group = 0, off_step = 0, bytes = 0;
};

// More tiles than any plan of such a range has (tiles are at least 1024
// samples): for callers that only want the kernel for many.
inline long matrix_tiles_at_most(int ndms, int t_processed)
{
    return (long)((ndms + 15) / 16) * ((t_processed + 1023) / 1024);
}

// Plan tables of one range over rows `pitch` bytes apart: fills `bytes` (when
// not null) as the kernel reads them and returns their layout; tile_out 0 when
// the range does not fit or the kernel it would replace is the better choice.
// planes 2: rows nchans .. 2 nchans - 1 hold the samples' high bytes.  Host
// only.
matrix_layout matrix_plan(const float* h_dmshifts, int nchans, int ndms, float mstartdm, float mdmstep, size_t pitch,
                          std::vector<uint8_t>* bytes, int planes = 1);

// Whether a 16-bit range of t samples is done sooner by the matrix kernel over
// byte planes (this layout) than by dedisperse_u16.
constexpr int kU16MatrixMinChannels = 24;
bool matrix_beats_u16(int nchans, long t, const matrix_layout& lay);

// p.pair_recs: the tables on the device.  planes 2: the sums are integers; a
// tile with a sum above 2^24, where the reference's float adds round, sets its
// entry of flags (n_dm_tiles x time tiles, time tile major; else 0) and has to
// be computed in channel order; more than half of over's 64 entries set flags
// every tile and computes none.  t_flags: the most samples (at least
// t_processed) that the rows hold for this range; the flags depend on them and
// not on t_processed.
hipError_t launch_dedisperse_matrix(const lds_params& p, const matrix_layout& lay, hipStream_t s,
                                    const int* over = nullptr, int* flags = nullptr, int t_flags = 0);

}  // namespace aa_hip

// Dedispersion of small ranges straight from the rows (see ddtr_rows.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "ddtr_matrix.h"

namespace aa_hip {

// Internal number of this kernel beside the LDS chunk shapes and the matrix
// kernel.
constexpr int kShapeRows = kShapeMatrix + 1;

// Whether a range of this size, alone on the device, is summed sooner straight
// from the rows than by the kernel it would have otherwise: the matrix kernel
// with this layout, or the chunk shape `variant` (-1: the direct kernel).
bool rows_beat_matrix(int nchans, int ndms, int t_processed, const matrix_layout& lay);
// Whether a range of a batch is done sooner by a matrix launch of its own than in
// the launch that its chunk shape `variant` shares with other ranges.
bool matrix_beats_shared(int nchans, int ndms, int t_processed, const matrix_layout& lay, int variant);
bool rows_beat_shape(int nchans, int ndms, int t_processed, int variant);

// Rows as for the LDS kernels (at whole dwords, 4 KiB readable past each row's
// longest window).
hipError_t launch_dedisperse_rows(const lds_params& p, hipStream_t s);

}  // namespace aa_hip

// Work-groups numbered from 0 on, in launches of any size: a launch runs at
// most 2^32 - 1 threads along x (HIP takes a larger one and runs a part of
// it), so the work-groups past that go along z.
#pragma once

#include <hip/hip_runtime.h>

namespace aa_hip {

// At least n work-groups of `threads` along x and z (the last ones may be too
// many: a kernel checks its number), `parts` along y.
inline dim3 linear_grid(long n, int threads, int parts = 1)
{
    const long most = (0xffffffffl / threads) & ~7l;   // a multiple of the XCDs
    if (n <= most) return dim3((unsigned)n, (unsigned)parts);
    return dim3((unsigned)most, (unsigned)parts, (unsigned)((n + most - 1) / most));
}

__device__ __forceinline__ long linear_block() { return (long)blockIdx.z * gridDim.x + blockIdx.x; }

}  // namespace aa_hip

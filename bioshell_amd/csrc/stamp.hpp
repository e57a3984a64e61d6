// stamp.hpp -- times of a call's stages, taken by its own kernels.
//
// An event record between two launches holds the stream for 5 to 6 us (two
// at the seam of two calls: 10 us; four per all-vs-all call: 22 us, more than
// the kernels of a small ensemble take).  Here the first work-group of a
// stage's first kernel, and the last work-group to finish of the call's last
// one, store the device's wall clock to device words that the host copies only
// when it is asked for times.  Per call: 200 x 76 FP64 25.4 -> 17.2 us, 2000 x
// 150 FP32 Gram 137 -> 122, 3001 x 187 with row statistics 126 -> 113, a query
// of 32 against 25,000 x 256 175 -> 156, 10,000 x 300 846 -> 832 (stores to
// pinned host words instead took 1 to 4 us more: each kernel then ends with
// a write across the host link).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bs {

// Device words of one call's clock; the last is its count of flagged pairs.
enum { kClkStart = 0, kClkMain = 1, kClkResolve = 2, kClkResolveEnd = 3, kClkEnd = 4, kClkCount = 5, kClkWords = 8 };

// The kernel starts (t may be null).
__device__ __forceinline__ void stamp_start(uint64_t* t)
{
    if (t && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *t = wall_clock64();
}

// A work-group ends; the last of them stamps.  `done` is a zero word that the
// launch leaves zero.  Every thread of the group calls it (t may be null).
__device__ __forceinline__ void stamp_end(uint64_t* t, unsigned* done)
{
    if (!t) return;
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(done, 1u) == gridDim.x * gridDim.y - 1) {
        *done = 0u;
        *t = wall_clock64();
    }
}

}  // namespace bs

// stamp.hpp -- times of a call's stages, taken by its own kernels.
//
// An event record between two launches holds the stream for 5 to 6 us (two
// at the seam of two calls: 10 us; four per all-vs-all call: 22 us, more than
// the kernels of a small ensemble take).  Here the first work-group of a
// stage's first kernel, and every work-group of the call's last one as it
// ends, store the device's wall clock to device words that the host copies only
// when it is asked for times.  Per call: 200 x 76 FP64 25.4 -> 17.2 us, 2000 x
// 150 FP32 Gram 137 -> 122, 3001 x 187 with row statistics 126 -> 113, a query
// of 32 against 25,000 x 256 175 -> 156, 10,000 x 300 846 -> 832 (stores to
// pinned host words instead took 1 to 4 us more: each kernel then ends with
// a write across the host link).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bs {

// Device words of one call's clock: its stages' times, its count of flagged
// pairs, and the words that the work-groups of its last launch share, each on a
// cache line of its own.  The call's end is the largest of kClkEnd and those;
// later calls only store larger times, so nothing is cleared between calls.
constexpr int kClkEndWords = 8, kClkEndStride = 16;
enum {
    kClkStart = 0, kClkMain = 1, kClkResolve = 2, kClkResolveEnd = 3, kClkEnd = 4, kClkCount = 5,
    kClkEnds = 16, kClkWords = kClkEnds + kClkEndWords * kClkEndStride
};

// The kernel starts (t may be null).
__device__ __forceinline__ void stamp_start(uint64_t* t)
{
    if (t && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *t = wall_clock64();
}

// The same in two parts: the time at the start and its store at the end, for
// kernels of one grid dimension that a store at the start makes slower (the
// per-pair kernels; FP32, 10,000 x 300: 9.19 ms with it, 9.03 this way, 9.06
// without any times).
__device__ __forceinline__ uint64_t stamp_read() { return blockIdx.x == 0 ? wall_clock64() : 0; }
__device__ __forceinline__ void stamp_store(uint64_t* t, uint64_t now)
{
    if (t && blockIdx.x == 0 && threadIdx.x == 0) *t = now;
}

// A work-group ends: `ends` (a clock's kClkEnds words, may be null) takes the
// later of its time and theirs.  Every thread of the group calls it.  An atomic
// without a result, which no wave waits for: counting the groups done on one
// word, so that the last one stamps, held a group's place until its turn came,
// 9 ns after the one before (FP32 per pair, 1000 x 20: 47.8 us; with no end
// taken 36.3; this way 36.7).  What is left is the wait for the group's stores;
// where its groups take equally long, a launch only has its last `tail`
// (kStampUniform: as many as the device holds at once) take part.
constexpr unsigned kStampUniform = 2048;
__device__ __forceinline__ void stamp_end(uint64_t* ends, unsigned tail = ~0u)
{
    const unsigned b = blockIdx.y * gridDim.x + blockIdx.x;
    if (!ends || gridDim.x * gridDim.y - b > tail) return;
    __syncthreads();
    if (threadIdx.x == 0)
        (void)atomicMax(reinterpret_cast<unsigned long long*>(ends + kClkEndStride * (b % kClkEndWords)),
                        (unsigned long long)wall_clock64());
}

}  // namespace bs

// cluster_rule.hpp -- the merging rules of hierarchical clustering, shared by
// the clustering kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace bs {

// The merging rules of strategies/mod.rs in f32, evaluated left to right with
// no contraction into fused multiply-adds (every operation rounds, as in the
// reference); the division is the correctly rounded f32 division.
__device__ inline float merge_rule(int rule, unsigned si, unsigned sj, unsigned sk, float dij,
                                   float dik, float djk)
{
#pragma clang fp contract(off)
    switch (rule) {
    case 0: return fminf(dik, djk);
    case 1: return fmaxf(dik, djk);
    case 2: {
        const float d = 1.0f / (float)(si + sj);
        return d * (float)si * dik + d * (float)sj * djk;
    }
    case 3: return 0.5f * dik + 0.5f * djk - 0.25f * dij;
    case 4: {
        const float d = 1.0f / (float)(si + sj);
        return d * (float)si * dik + d * (float)sj * djk - (float)si * (float)sj * d * d * dij;
    }
    default: {
        const float d = 1.0f / (float)(si + sj + sk);
        return d * (float)(si + sk) * dik + d * (float)(sj + sk) * djk - (float)sk * d * dij;
    }
    }
}

}  // namespace bs

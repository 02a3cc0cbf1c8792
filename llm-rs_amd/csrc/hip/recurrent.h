// The formulas of the recurrent mixers that the scans (recurrent.hip) and the products of single tokens (gemm_few.hip) share.
#pragma once
#include "common.h"

#define LOG2_E 1.44269504088896341f

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f32(float x) { return x > 20.0f ? x : log1pf(expf(x)); }
// minGRU's new state from the old one, the gate z and the candidate's sum u (see recurrent.hip)
__device__ __forceinline__ float mingru_state(float s, float z, float u) {
    const float cand = u >= 0.0f ? u + 0.5f : sigmoid_f32(u);
    return (1.0f - z) * s + z * cand;
}

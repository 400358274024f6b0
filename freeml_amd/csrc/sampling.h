// Sampled picks (fmlh_nanollm_set_sampling): what the graph path's kernel and the relay kernel's
// lm_head role share.
#pragma once

#include "fmlh_internal.h"

namespace fmlh {

struct SampleCfg {
    float inv_temp = 0.0f;
    int top_k = 0;
    unsigned long long seed = 0;
    bool on = false;  // false: greedy
};

__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ float sample_uniform(unsigned long long seed, int b, int p) {
    const unsigned long long key = ((unsigned long long)(unsigned)b << 32) | (unsigned)p;
    return (float)(splitmix64(seed ^ splitmix64(key)) >> 40) * (1.0f / 16777216.0f);
}

// Order-preserving float -> uint32 (larger float, larger key; -0 and +0 distinct, no NaNs).
__device__ __forceinline__ uint32_t float_key(float v) {
    const uint32_t u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

}  // namespace fmlh

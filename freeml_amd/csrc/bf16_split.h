// Exact split of fp32 values into three bf16 parts (device code): x = x0 + x1 + x2, each the
// round-to-nearest bf16 of what is left.
#pragma once

#include "fmlh_internal.h"

namespace fmlh {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{x, y}, bf16x2));
}

// Eight floats, times `scale`, -> their three bf16 planes (one 16-byte unit each).
__device__ __forceinline__ void split8(const float (&v)[8], uintx4 (&p)[3], float scale = 1.0f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = v[2 * i] * scale, y = v[2 * i + 1] * scale;
        const uint32_t p0 = pack_bf16(x, y);
        const float rx = x - __uint_as_float(p0 << 16), ry = y - __uint_as_float(p0 & 0xffff0000u);
        const uint32_t p1 = pack_bf16(rx, ry);
        const float sx = rx - __uint_as_float(p1 << 16), sy = ry - __uint_as_float(p1 & 0xffff0000u);
        p[0][i] = p0;
        p[1][i] = p1;
        p[2][i] = pack_bf16(sx, sy);
    }
}

// The part products of a b that are 2^-16 of it or more, smallest first: a[kSplitA[q]] b[kSplitB[q]].
constexpr int kSplitA[6] = {2, 1, 0, 1, 0, 0}, kSplitB[6] = {0, 1, 2, 0, 1, 0};

}  // namespace
}  // namespace fmlh

// fp32 products on the bf16 matrix cores (gemm_split.hip).
#pragma once

#include "fmlh_internal.h"

namespace fmlh {

// C = A op(B) per plane, with A M x K rows (a_kc: K contiguous, row stride lda) or stored K x M
// (rows contiguous, stride lda between k), B likewise as N x K (b_kc) or K x N.
struct SplitGemm {
    const float* A = nullptr;
    int lda = 0;
    bool a_kc = true;
    size_t a_plane = 0;
    const float* B = nullptr;
    int ldb = 0;
    bool b_kc = true;
    size_t b_plane = 0;
    float* C = nullptr;
    int ldc = 0;
    size_t c_plane = 0;
    int M = 0, N = 0, K = 0, planes = 1;
    int epi = kEpiNone;  // a_kc only, one plane
    const float* R = nullptr;
    int ldr = 0;
    KvDest kv;  // kEpiKV only
    // splits > 1 (a_kc, one plane): partial sums over K ranges of k_per_split (a multiple of 16)
    // go to partial[split][M][N] instead of C, without an epilogue.
    int splits = 1, k_per_split = 0;
    float* partial = nullptr;
    int tile = 128;    // 128 x 128 or 64 x 64 tiles
    int k_groups = 1;  // 64: waves per work-group twofold, each half on half of K
    hipStream_t s = nullptr;
};

// Whether strides and alignment allow it (any M, N, K).
bool gemm_split_takes(const SplitGemm& g);
int gemm_split(const SplitGemm& g);

}  // namespace fmlh

// GEMM kernels behind Mul / MatMul_Strided and the token loop's projections.
//
//  * gemm_split_kernel (gemm_split.hip): everything wider than the batched decode, each fp32
//    operand split into three bf16 parts on the bf16 matrix cores.
//  * gemm_mfma_kernel: fp32 MFMA tiles (v_mfma_f32_32x32x2f32) with register-staged,
//    double-buffered LDS, for either B layout: 8 < M <= 64 (batched decode), the smallest
//    products above, and row strides past the split tiles' 32-bit offsets.  Optional split-K
//    writes partial sums that splitk_reduce_kernel adds in a fixed order (deterministic) before
//    the epilogue.
//  * skinny kernels for M <= 8 (single-sequence decode): HBM-bound weight streaming, every
//    weight read once, all M rows accumulated per weight load.
//  * gemm_strided_kernel: any transpose mode and element strides (MatMul_Strided views).
//
// All products accumulate in fp32.  The reference (MatrixBase_Mul.h:521-545) sums each output
// sequentially over k; these kernels sum in other orders, so results differ from it by fp32
// rounding only (compared with a tolerance in the parity tests).
#include "fmlh_internal.h"
#include "gemm_split.h"

#include <algorithm>
#include <cstdio>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>

namespace fmlh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float gelu_ref(float x) {
    return 0.5f * x * (1.0f + erff(x / 1.41421354f));
}

template <int EPI>
__device__ __forceinline__ float epilogue(float acc, const float* R, size_t ridx) {
    if constexpr (EPI == kEpiGelu) return gelu_ref(acc);
    else if constexpr (EPI == kEpiResid) return R[ridx] + acc;
    else return acc;
}

// ---------------------------------------------------------------------------------------
// MFMA tile kernel.
//
// v_mfma_f32_32x32x2f32 operand layout (one 64-lane wave, h = lane / 32, c = lane % 32):
//   A (32 x 2):  lane supplies A[c][h]          B (2 x 32): lane supplies B[h][c]
//   D (32 x 32): lane holds D[8*(r/4) + 4*h + r%4][c] in accumulator register r.
// Within a 16-wide K block the k index of MFMA step s for half h is 8*h + s, so each lane
// reads 8 consecutive k values of its A row / B column from LDS (two 16-byte reads).
// ---------------------------------------------------------------------------------------
constexpr int KB = 16;       // K block
constexpr int LDS_STRIDE = KB + 4;  // floats per LDS row (padding spreads banks)

template <int BM, int BN, bool BT, int EPI, bool SPLIT>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
    float* __restrict__ C, int ldc, int M, int N, int K, const float* R, int ldr,
    float* __restrict__ partial, int k_per_split) {
    static_assert(BM % 64 == 0 && BN % 64 == 0, "tile must be a multiple of 64");
    constexpr int WM = BM / 2, WN = BN / 2;       // wave tile (2 x 2 waves)
    constexpr int MB = WM / 32, NB = WN / 32;     // 32x32 blocks per wave
    constexpr int A_F4 = BM * KB / 4 / 256;       // float4 loads per thread per K block
    constexpr int B_F4 = BN * KB / 4 / 256;

    __shared__ float As[2][BM][LDS_STRIDE];
    __shared__ float Bs[2][BN][LDS_STRIDE];

    const int tid = threadIdx.x;
    const int lane = tid % 64, wave = tid / 64;
    const int wm = wave / 2, wn = wave % 2;
    const int h = lane / 32, c = lane % 32;
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    const int kbeg = SPLIT ? blockIdx.z * k_per_split : 0;
    const int kend = SPLIT ? min(K, kbeg + k_per_split) : K;

    floatx16 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    floatx4 ra[A_F4], rb[B_F4];

    auto load_global = [&](int k0) {
#pragma unroll
        for (int t = 0; t < A_F4; ++t) {
            const int idx = tid + t * 256;          // BM rows x 4 float4
            const int r = idx / 4, q = idx % 4;
            const int gr = row0 + r;
            ra[t] = (gr < M) ? *reinterpret_cast<const floatx4*>(A + (size_t)gr * lda + k0 + 4 * q)
                             : floatx4{0.f, 0.f, 0.f, 0.f};
        }
        if constexpr (BT) {  // B stored N x K: rows of the tile are output columns
#pragma unroll
            for (int t = 0; t < B_F4; ++t) {
                const int idx = tid + t * 256;
                const int r = idx / 4, q = idx % 4;
                const int gc = col0 + r;
                rb[t] = (gc < N) ? *reinterpret_cast<const floatx4*>(B + (size_t)gc * ldb + k0 + 4 * q)
                                 : floatx4{0.f, 0.f, 0.f, 0.f};
            }
        } else {  // B stored K x N: the tile is KB rows of BN contiguous floats
#pragma unroll
            for (int t = 0; t < B_F4; ++t) {
                const int idx = tid + t * 256;
                const int kr = idx / (BN / 4), q = idx % (BN / 4);
                const int gc = col0 + 4 * q;
                const float* src = B + (size_t)(k0 + kr) * ldb + gc;
                if (gc + 3 < N) {
                    rb[t] = *reinterpret_cast<const floatx4*>(src);
                } else {
                    floatx4 v = {0.f, 0.f, 0.f, 0.f};
                    for (int e = 0; e < 4; ++e)
                        if (gc + e < N) v[e] = src[e];
                    rb[t] = v;
                }
            }
        }
    };

    auto store_lds = [&](int buf) {
#pragma unroll
        for (int t = 0; t < A_F4; ++t) {
            const int idx = tid + t * 256;
            const int r = idx / 4, q = idx % 4;
            *reinterpret_cast<floatx4*>(&As[buf][r][4 * q]) = ra[t];
        }
        if constexpr (BT) {
#pragma unroll
            for (int t = 0; t < B_F4; ++t) {
                const int idx = tid + t * 256;
                const int r = idx / 4, q = idx % 4;
                *reinterpret_cast<floatx4*>(&Bs[buf][r][4 * q]) = rb[t];
            }
        } else {
#pragma unroll
            for (int t = 0; t < B_F4; ++t) {
                const int idx = tid + t * 256;
                const int kr = idx / (BN / 4), q = idx % (BN / 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) Bs[buf][4 * q + e][kr] = rb[t][e];
            }
        }
    };

    int buf = 0;
    if (kbeg < kend) {
        load_global(kbeg);
        store_lds(0);
    }
    __syncthreads();
    for (int k0 = kbeg; k0 < kend; k0 += KB) {
        const bool more = k0 + KB < kend;
        if (more) load_global(k0 + KB);
        floatx4 a_lo[MB], a_hi[MB], b_lo[NB], b_hi[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const float* p = &As[buf][wm * WM + i * 32 + c][8 * h];
            a_lo[i] = *reinterpret_cast<const floatx4*>(p);
            a_hi[i] = *reinterpret_cast<const floatx4*>(p + 4);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const float* p = &Bs[buf][wn * WN + j * 32 + c][8 * h];
            b_lo[j] = *reinterpret_cast<const floatx4*>(p);
            b_hi[j] = *reinterpret_cast<const floatx4*>(p + 4);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const float av = s < 4 ? a_lo[i][s] : a_hi[i][s - 4];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const float bv = s < 4 ? b_lo[j][s] : b_hi[j][s - 4];
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[i][j], 0, 0, 0);
                }
            }
        }
        if (more) store_lds(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }

#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int gc = col0 + wn * WN + j * 32 + c;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int gr = row0 + wm * WM + i * 32 + 8 * (r / 4) + 4 * h + (r % 4);
                if (gr < M && gc < N) {
                    if constexpr (SPLIT) {
                        partial[((size_t)blockIdx.z * M + gr) * N + gc] = acc[i][j][r];
                    } else {
                        C[(size_t)gr * ldc + gc] =
                            epilogue<EPI>(acc[i][j][r], R, (size_t)gr * ldr + gc);
                    }
                }
            }
        }
    }
}

// Adds the split partial sums in split order, then applies the epilogue.
template <int EPI>
__global__ void splitk_reduce_kernel(const float* __restrict__ partial, int splits, float* C,
                                     int ldc, int M, int N, const float* R, int ldr) {
    const size_t total = (size_t)M * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total;
         i += (size_t)gridDim.x * blockDim.x) {
        float s = 0.0f;
        for (int z = 0; z < splits; ++z) s += partial[(size_t)z * total + i];
        const size_t r = i / N, col = i % N;
        C[r * ldc + col] = epilogue<EPI>(s, R, r * ldr + col);
    }
}

// ---------------------------------------------------------------------------------------
// Split-K NT kernel for short K ranges (batched decode: M <= 64 rows, K-range of at most
// kNtSplitMaxBlocks 16-wide blocks per work-group).  The whole range of both 64 x 64 tiles is
// copied into LDS at once (one stage per block), so the work-group waits for global memory
// once instead of once per block; then every MFMA runs back to back.  Writes the partial sums
// of split blockIdx.z to partial[z][M][N] (added up by the caller).  Same operand layout and
// k order as gemm_mfma_kernel.
// ---------------------------------------------------------------------------------------
constexpr int kNtSplitMaxBlocks = 8;

// Float4 q of a 16-float row r is stored at q ^ quad_swz(r), which puts the operand reads of any 8
// or 16 consecutive lanes (one row each, same q) on distinct banks (a direct-to-LDS copy fills
// LDS contiguously, so rows cannot be padded).
__device__ __forceinline__ int quad_swz(int r) { return ((r >> 1) ^ ((r >> 3) & 1)) & 3; }

__global__ __launch_bounds__(256) void gemm_nt_split_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, int M, int N,
    int k_per_split, float* __restrict__ partial) {
    constexpr int BM = 64, BN = 64, A_FL = BM * KB, ST_FL = (BM + BN) * KB;
    extern __shared__ __attribute__((aligned(16))) float nts_lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int h = lane >> 5, c = lane & 31;
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    const int kbeg = blockIdx.z * k_per_split;
    const int nk = k_per_split / KB;  // <= kNtSplitMaxBlocks (host check)

    const int crow = lane >> 2;
    const int cq = (lane & 3) ^ quad_swz(crow);
    const float* asrc = A + (size_t)min(row0 + 16 * wave + crow, M - 1) * lda + kbeg + 4 * cq;
    const float* bsrc = B + (size_t)min(col0 + 16 * wave + crow, N - 1) * ldb + kbeg + 4 * cq;
    for (int kb = 0; kb < nk; ++kb) {
        float* sa = nts_lds + kb * ST_FL;
        copy16_to_lds(sa + wave * 256, asrc + kb * KB);
        copy16_to_lds(sa + A_FL + wave * 256, bsrc + kb * KB);
    }
    const int p0 = (2 * h) ^ quad_swz(c);
    const int p1 = p0 ^ 1;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    copies_barrier<0>();
    for (int kb = 0; kb < nk; ++kb) {
        const float* sa = nts_lds + kb * ST_FL + (wm * 32 + c) * KB;
        const float* sb = nts_lds + kb * ST_FL + A_FL + (wn * 32 + c) * KB;
        const floatx4 a_lo = *reinterpret_cast<const floatx4*>(sa + 4 * p0);
        const floatx4 b_lo = *reinterpret_cast<const floatx4*>(sb + 4 * p0);
        const floatx4 a_hi = *reinterpret_cast<const floatx4*>(sa + 4 * p1);
        const floatx4 b_hi = *reinterpret_cast<const floatx4*>(sb + 4 * p1);
#pragma unroll
        for (int s = 0; s < 8; ++s)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s < 4 ? a_lo[s] : a_hi[s - 4],
                                                       s < 4 ? b_lo[s] : b_hi[s - 4], acc, 0, 0, 0);
    }
    const int gc = col0 + wn * 32 + c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int gr = row0 + wm * 32 + 8 * (r / 4) + 4 * h + (r % 4);
        if (gr < M && gc < N) partial[((size_t)blockIdx.z * M + gr) * N + gc] = acc[r];
    }
}

// ---------------------------------------------------------------------------------------
// Skinny kernels (M <= 8).
// ---------------------------------------------------------------------------------------
constexpr int SK_MAXM = 8;
constexpr int SK_KCHUNK = 16;  // k rows per block of the NN kernel

// NN: B is K x N.  Block (x = 256-column strip, y = k chunk); lane owns 4 columns.  Writes
// partial[y][m][n]; splitk_reduce_kernel sums the chunks in order and applies the epilogue.
__global__ __launch_bounds__(64) void skinny_nn_partial_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
    float* __restrict__ partial, int M, int N, int K) {
    const int col = blockIdx.x * 256 + threadIdx.x * 4;
    const int k0 = blockIdx.y * SK_KCHUNK;
    const int k1 = min(K, k0 + SK_KCHUNK);
    if (col >= N) return;
    float acc[SK_MAXM][4];
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[m][e] = 0.0f;
    const bool full = col + 3 < N;
    for (int k = k0; k < k1; ++k) {
        floatx4 w;
        const float* src = B + (size_t)k * ldb + col;
        if (full) {
            w = *reinterpret_cast<const floatx4*>(src);
        } else {
            w = floatx4{0.f, 0.f, 0.f, 0.f};
            for (int e = 0; e < 4; ++e)
                if (col + e < N) w[e] = src[e];
        }
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m) {
            if (m < M) {
                const float a = A[(size_t)m * lda + k];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][e] += a * w[e];
            }
        }
    }
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m) {
        if (m < M) {
            float* dst = partial + ((size_t)blockIdx.y * M + m) * N + col;
            for (int e = 0; e < 4; ++e)
                if (col + e < N) dst[e] = acc[m][e];
        }
    }
}

// NT: B is N x K (rows contiguous in k).  16 lanes per output column n, 4 columns per wave.
template <int EPI>
__global__ __launch_bounds__(64) void skinny_nt_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, float* C, int ldc,
    int M, int N, int K, const float* R, int ldr) {
    const int sub = threadIdx.x % 16;
    const int n = blockIdx.x * 4 + threadIdx.x / 16;
    float acc[SK_MAXM];
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m) acc[m] = 0.0f;
    if (n < N) {
        const float* w = B + (size_t)n * ldb;
        for (int k = sub * 4; k < K; k += 64) {
            const floatx4 wv = *reinterpret_cast<const floatx4*>(w + k);
#pragma unroll
            for (int m = 0; m < SK_MAXM; ++m) {
                if (m < M) {
                    const floatx4 av = *reinterpret_cast<const floatx4*>(A + (size_t)m * lda + k);
                    acc[m] += av[0] * wv[0] + av[1] * wv[1] + av[2] * wv[2] + av[3] * wv[3];
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m) {
        float v = acc[m];
        v += __shfl_xor(v, 8, 16);
        v += __shfl_xor(v, 4, 16);
        v += __shfl_xor(v, 2, 16);
        v += __shfl_xor(v, 1, 16);
        acc[m] = v;
    }
    if (n < N && sub == 0) {
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m)
            if (m < M) C[(size_t)m * ldc + n] = epilogue<EPI>(acc[m], R, (size_t)m * ldr + n);
    }
}

// NT, KS waves per output column (KS = 1, 2 or 4): wave j of a column takes float4 chunks
// j, j + KS, ... of each 64-chunk stretch of K (its 64 lanes side by side, four chunks in flight
// per lane) and keeps the M <= 8 row partials; a wave reduction, then the KS waves' sums added in
// wave order through LDS.  4 / KS columns per work-group: small N (the residual projections,
// N = C) still spreads over every CU.
// LN: A holds rows before a LayerNorm; the work-group first forms each row's mean and 1/std
// exactly as layernorm_kernel does (wave per row, lane l holding elements l + 64 i, two-pass
// variance), then normalises the A values it loads: ((a - mean) * inv_std) * gamma + beta.
constexpr int kSkLnNE = 16;  // row elements per lane of the statistics pass (K <= 1024)

template <int EPI, int KS, bool LN = false>
__global__ __launch_bounds__(256) void skinny_nt_wave_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, float* C, int ldc,
    int M, int N, int K, const float* R, int ldr, const float* __restrict__ ln_g = nullptr,
    const float* __restrict__ ln_b = nullptr, float ln_eps = 0.0f) {
    constexpr int CPW = 4 / KS;  // columns per work-group
    __shared__ float part[4][SK_MAXM];
    __shared__ float ln_st[LN ? SK_MAXM : 1][2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = wave / KS, j = wave % KS;
    const int n = blockIdx.x * CPW + col;
    if constexpr (LN) {
        const float inv_cols = 1.0f / (float)K;
        for (int m = wave; m < M; m += 4) {
            const float* xr = A + (size_t)m * lda;
            float v[kSkLnNE];
#pragma unroll
            for (int i = 0; i < kSkLnNE; ++i) {
                const int c = lane + 64 * i;
                v[i] = c < K ? xr[c] : 0.0f;
            }
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < kSkLnNE; ++i)
                if (lane + 64 * i < K) sum += v[i];
            const float mean = wave_sum(sum) * inv_cols;
            float q = 0.0f;
#pragma unroll
            for (int i = 0; i < kSkLnNE; ++i)
                if (lane + 64 * i < K) {
                    const float d = v[i] - mean;
                    q += d * d;
                }
            const float inv_std = 1.0f / sqrtf(wave_sum(q) * inv_cols + ln_eps);
            if (lane == 0) {
                ln_st[m][0] = mean;
                ln_st[m][1] = inv_std;
            }
        }
        __syncthreads();
    }
    // The residual's values are loaded now, so the store does not wait for another round trip.
    float rv[SK_MAXM];
    if constexpr (EPI == kEpiResid) {
        if (n < N && j == 0 && lane == 0) {
#pragma unroll
            for (int m = 0; m < SK_MAXM; ++m) rv[m] = m < M ? R[(size_t)m * ldr + n] : 0.0f;
        }
    }
    float acc[SK_MAXM];
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m) acc[m] = 0.0f;
    if (n < N) {
        const float* w = B + (size_t)n * ldb;
        const int nch = K / 4;
#pragma unroll 4
        for (int e = lane + 64 * j; e < nch; e += 64 * KS) {
            const floatx4 wv = *reinterpret_cast<const floatx4*>(w + 4 * e);
            floatx4 gv, bv;
            if constexpr (LN) {
                gv = *reinterpret_cast<const floatx4*>(ln_g + 4 * e);
                if (ln_b) bv = *reinterpret_cast<const floatx4*>(ln_b + 4 * e);
                else bv = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int m = 0; m < SK_MAXM; ++m) {
                if (m < M) {
                    floatx4 av = *reinterpret_cast<const floatx4*>(A + (size_t)m * lda + 4 * e);
                    if constexpr (LN) {
                        const float mean = ln_st[m][0], inv_std = ln_st[m][1];
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const float nrm = (av[t] - mean) * inv_std;
                            av[t] = nrm * gv[t] + bv[t];
                        }
                    }
                    acc[m] += av[0] * wv[0] + av[1] * wv[1] + av[2] * wv[2] + av[3] * wv[3];
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < SK_MAXM; ++m)
        if (m < M) acc[m] = wave_sum(acc[m]);
    if constexpr (KS > 1) {
        if (lane == 0) {
#pragma unroll
            for (int m = 0; m < SK_MAXM; ++m) part[wave][m] = acc[m];
        }
        __syncthreads();
        if (j == 0) {
#pragma unroll
            for (int m = 0; m < SK_MAXM; ++m) {
                float t = part[wave][m];
#pragma unroll
                for (int q = 1; q < KS; ++q) t += part[wave + q][m];
                acc[m] = t;
            }
        }
    }
    if (n < N && j == 0 && lane == 0) {
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m) {
            if (m < M) {
                if constexpr (EPI == kEpiResid) C[(size_t)m * ldc + n] = rv[m] + acc[m];
                else C[(size_t)m * ldc + n] = epilogue<EPI>(acc[m], R, (size_t)m * ldr + n);
            }
        }
    }
}

// Wide products (N > 4096, e.g. a 50304-row lm_head): one wave per group of NC columns, so
// every activation float4 the wave loads serves NC weight rows (with one column per wave the
// M <= 8 activation rows are re-read from the caches once per column: ~8x the weight bytes).
// Per column the arithmetic is that of skinny_nt_wave_kernel with KS = 1.
template <int EPI, int NC>
__global__ __launch_bounds__(256) void skinny_nt_wide_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, float* C, int ldc,
    int M, int N, int K, const float* R, int ldr) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * 4 + wave) * NC;
    if (n0 >= N) return;  // wave-uniform; no barrier follows
    const float* w[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) w[c] = B + (size_t)min(n0 + c, N - 1) * ldb;
    float acc[NC][SK_MAXM];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m) acc[c][m] = 0.0f;
    const int nch = K / 4;
#pragma unroll 2
    for (int e = lane; e < nch; e += 64) {
        floatx4 wv[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) wv[c] = *reinterpret_cast<const floatx4*>(w[c] + 4 * e);
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m) {
            if (m < M) {
                const floatx4 av = *reinterpret_cast<const floatx4*>(A + (size_t)m * lda + 4 * e);
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    acc[c][m] += av[0] * wv[c][0] + av[1] * wv[c][1] + av[2] * wv[c][2] + av[3] * wv[c][3];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int m = 0; m < SK_MAXM; ++m)
            if (m < M) acc[c][m] = wave_sum(acc[c][m]);
    if (lane == 0) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int n = n0 + c;
            if (n < N) {
#pragma unroll
                for (int m = 0; m < SK_MAXM; ++m)
                    if (m < M) C[(size_t)m * ldc + n] = epilogue<EPI>(acc[c][m], R, (size_t)m * ldr + n);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------
// Generic strided product: C[i*o_rs + j*o_cs] = sum_k A(i,k) B(k,j), batched over planes.
// A(i,k) = L[i*l_rs + k*l_cs] (TL: L[k*l_rs + i*l_cs]); B(k,j) = R[k*r_rs + j*r_cs]
// (TR: R[j*r_rs + k*r_cs]).  The callers are FreeML's per-head attention products and the
// Dense weight gradients (Mul<Left>): small outputs (e.g. 256 x 64) over K of a few hundred,
// so the tile is 32 x 32 (more work-groups per product) and K is staged in chunks of 64 with
// the next chunk's loads in flight (registers) while the current one is multiplied from LDS.
// Each thread loads with the strided operand's contiguous index fastest across threads.
// ---------------------------------------------------------------------------------------
constexpr uint32_t kStT = 32, kStKC = 64, kStPer = kStT * kStKC / 256;

template <bool TL, bool TR>
__global__ __launch_bounds__(256) void gemm_strided_kernel(
    float* __restrict__ out, const float* __restrict__ L, const float* __restrict__ Rm,
    uint32_t M, uint32_t N, uint32_t K, uint32_t l_rs, uint32_t l_cs, uint32_t r_rs,
    uint32_t r_cs, uint32_t o_rs, uint32_t o_cs, size_t l_plane, size_t r_plane,
    size_t o_plane) {
    __shared__ float As[kStKC][kStT + 1];  // As[k][i]
    __shared__ float Bs[kStKC][kStT + 1];  // Bs[k][j]
    const float* Lp = L + blockIdx.z * l_plane;
    const float* Rp = Rm + blockIdx.z * r_plane;
    float* Op = out + blockIdx.z * o_plane;
    const uint32_t row0 = blockIdx.y * kStT, col0 = blockIdx.x * kStT;
    const uint32_t t = threadIdx.x;
    // Element e = t + 256 r of a chunk: (i, k) of A and (k, j) of B.
    auto a_ik = [&](uint32_t e, uint32_t& i, uint32_t& k) {
        if (TL) { i = e % kStT; k = e / kStT; } else { k = e % kStKC; i = e / kStKC; }
    };
    auto b_kj = [&](uint32_t e, uint32_t& k, uint32_t& j) {
        if (TR) { k = e % kStKC; j = e / kStKC; } else { j = e % kStT; k = e / kStT; }
    };
    float ra[kStPer], rb[kStPer];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t r = 0; r < kStPer; ++r) {
            uint32_t i, k, j, kb;
            a_ik(t + 256 * r, i, k);
            b_kj(t + 256 * r, kb, j);
            const uint32_t gi = row0 + i, gk = k0 + k, gj = col0 + j, gkb = k0 + kb;
            ra[r] = (gi < M && gk < K)
                        ? (TL ? Lp[(size_t)gk * l_rs + (size_t)gi * l_cs] : Lp[(size_t)gi * l_rs + (size_t)gk * l_cs])
                        : 0.0f;
            rb[r] = (gj < N && gkb < K)
                        ? (TR ? Rp[(size_t)gj * r_rs + (size_t)gkb * r_cs] : Rp[(size_t)gkb * r_rs + (size_t)gj * r_cs])
                        : 0.0f;
        }
    };
    const uint32_t tx = t % 16, ty = t / 16;  // outputs (2 ty + a, 2 tx + b)
    float acc[2][2] = {};
    load(0);
    for (uint32_t k0 = 0; k0 < K; k0 += kStKC) {
        __syncthreads();  // the previous chunk has been read out of LDS
#pragma unroll
        for (uint32_t r = 0; r < kStPer; ++r) {
            uint32_t i, k, j, kb;
            a_ik(t + 256 * r, i, k);
            b_kj(t + 256 * r, kb, j);
            As[k][i] = ra[r];
            Bs[kb][j] = rb[r];
        }
        __syncthreads();
        if (k0 + kStKC < K) load(k0 + kStKC);
#pragma unroll 16
        for (uint32_t kk = 0; kk < kStKC; ++kk) {
            const float a0 = As[kk][2 * ty], a1 = As[kk][2 * ty + 1];
            const float b0 = Bs[kk][2 * tx], b1 = Bs[kk][2 * tx + 1];
            acc[0][0] += a0 * b0;
            acc[0][1] += a0 * b1;
            acc[1][0] += a1 * b0;
            acc[1][1] += a1 * b1;
        }
    }
#pragma unroll
    for (uint32_t a = 0; a < 2; ++a) {
        const uint32_t gi = row0 + 2 * ty + a;
#pragma unroll
        for (uint32_t b = 0; b < 2; ++b) {
            const uint32_t gj = col0 + 2 * tx + b;
            if (gi < M && gj < N) Op[(size_t)gi * o_rs + (size_t)gj * o_cs] = acc[a][b];
        }
    }
}

// Same product for K > kStKC: the work-group's four waves each take one K chunk of every pass
// (pass = 4 chunks) for the same TT x TT output tile, with the next pass's operands in flight
// during the multiply; the four partial tiles are then added in wave order (deterministic).
// TT = 16 (chunk 64) spreads small outputs over more work-groups -- a 256 x 64 per-head
// product with K = 256 becomes 64 work-groups that each load all of K at once -- and TT = 32
// (chunk 32) serves larger outputs.  Lane (tx, ty) = (lane % 8, lane / 8) holds the
// MT x MT outputs (MT ty + x, MT tx + y), MT = TT / 8.
constexpr uint32_t kWsWaves = 4;

template <uint32_t MT> struct VecOf;
template <> struct VecOf<2> { using type = float2; };
template <> struct VecOf<4> { using type = float4; };

template <bool TL, bool TR, uint32_t TT>
__global__ __launch_bounds__(256) void gemm_strided_wsplit_kernel(
    float* __restrict__ out, const float* __restrict__ L, const float* __restrict__ Rm,
    uint32_t M, uint32_t N, uint32_t K, uint32_t l_rs, uint32_t l_cs, uint32_t r_rs,
    uint32_t r_cs, uint32_t o_rs, uint32_t o_cs, size_t l_plane, size_t r_plane,
    size_t o_plane) {
    constexpr uint32_t KC = 1024 / TT;        // K chunk per wave
    constexpr uint32_t LD = TT + 4;           // LDS row stride (rows stay 16-byte aligned)
    constexpr uint32_t PER = TT * KC / kWave;  // elements per lane per operand (16)
    constexpr uint32_t MT = TT / 8;           // lane micro-tile
    using Vec = typename VecOf<MT>::type;
    static_assert(TT * TT <= 2 * KC * LD, "partial tile must fit the wave's LDS slice");
    __shared__ __attribute__((aligned(16))) float sm[kWsWaves][2 * KC * LD];
    const float* Lp = L + blockIdx.z * l_plane;
    const float* Rp = Rm + blockIdx.z * r_plane;
    float* Op = out + blockIdx.z * o_plane;
    const uint32_t row0 = blockIdx.y * TT, col0 = blockIdx.x * TT;
    const uint32_t lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    float* As = sm[w];            // As[k * LD + i]
    float* Bs = sm[w] + KC * LD;  // Bs[k * LD + j]
    auto a_ik = [&](uint32_t e, uint32_t& i, uint32_t& k) {
        if (TL) { i = e % TT; k = e / TT; } else { k = e % KC; i = e / KC; }
    };
    auto b_kj = [&](uint32_t e, uint32_t& k, uint32_t& j) {
        if (TR) { k = e % KC; j = e / KC; } else { j = e % TT; k = e / TT; }
    };
    float ra[PER], rb[PER];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t r = 0; r < PER; ++r) {
            uint32_t i, k, j, kb;
            a_ik(lane + kWave * r, i, k);
            b_kj(lane + kWave * r, kb, j);
            const uint32_t gi = row0 + i, gk = k0 + k, gj = col0 + j, gkb = k0 + kb;
            ra[r] = (gi < M && gk < K)
                        ? (TL ? Lp[(size_t)gk * l_rs + (size_t)gi * l_cs] : Lp[(size_t)gi * l_rs + (size_t)gk * l_cs])
                        : 0.0f;
            rb[r] = (gj < N && gkb < K)
                        ? (TR ? Rp[(size_t)gj * r_rs + (size_t)gkb * r_cs] : Rp[(size_t)gkb * r_rs + (size_t)gj * r_cs])
                        : 0.0f;
        }
    };
    const uint32_t tx = lane % 8, ty = lane / 8;
    float acc[MT][MT] = {};
    constexpr uint32_t kPass = kWsWaves * KC;
    load(w * KC);
    for (uint32_t kp = 0; kp < K; kp += kPass) {
        __syncthreads();  // this wave's previous chunk has been read out of LDS
#pragma unroll
        for (uint32_t r = 0; r < PER; ++r) {
            uint32_t i, k, j, kb;
            a_ik(lane + kWave * r, i, k);
            b_kj(lane + kWave * r, kb, j);
            As[k * LD + i] = ra[r];
            Bs[kb * LD + j] = rb[r];
        }
        __syncthreads();
        if (kp + kPass < K) load(kp + kPass + w * KC);
#pragma unroll 8
        for (uint32_t kk = 0; kk < KC; ++kk) {
            const Vec a = *reinterpret_cast<const Vec*>(&As[kk * LD + MT * ty]);
            const Vec b = *reinterpret_cast<const Vec*>(&Bs[kk * LD + MT * tx]);
            const float* av = reinterpret_cast<const float*>(&a);
            const float* bv = reinterpret_cast<const float*>(&b);
#pragma unroll
            for (uint32_t x = 0; x < MT; ++x)
#pragma unroll
                for (uint32_t y = 0; y < MT; ++y) acc[x][y] += av[x] * bv[y];
        }
    }
    __syncthreads();
    float* part = sm[w];  // this wave's TT x TT partial tile, row-major
#pragma unroll
    for (uint32_t x = 0; x < MT; ++x)
#pragma unroll
        for (uint32_t y = 0; y < MT; ++y) part[(MT * ty + x) * TT + MT * tx + y] = acc[x][y];
    __syncthreads();
    for (uint32_t idx = threadIdx.x; idx < TT * TT; idx += 256) {
        const uint32_t i = idx / TT, j = idx % TT;
        float v = sm[0][idx];
#pragma unroll
        for (uint32_t ww = 1; ww < kWsWaves; ++ww) v += sm[ww][idx];
        const uint32_t gi = row0 + i, gj = col0 + j;
        if (gi < M && gj < N) Op[(size_t)gi * o_rs + (size_t)gj * o_cs] = v;
    }
}

// Process-wide split-K workspace for callers that do not bring their own.
std::mutex g_ws_mu;
float* g_ws = nullptr;
size_t g_ws_elems = 0;

int global_workspace(size_t elems, float** ws) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    if (elems > g_ws_elems) {
        if (g_ws) {
            FMLH_HIP(hipStreamSynchronize(stream()));
            FMLH_HIP(hipFree(g_ws));
            g_ws = nullptr;
            g_ws_elems = 0;
        }
        FMLH_TRY(device_malloc(reinterpret_cast<void**>(&g_ws), elems * sizeof(float)));
        g_ws_elems = elems;
    }
    *ws = g_ws;
    return FMLH_OK;
}

template <int EPI>
int launch_reduce(const float* partial, int splits, float* C, int ldc, int M, int N,
                  const float* R, int ldr, hipStream_t s) {
    const size_t total = (size_t)M * N;
    hipLaunchKernelGGL(splitk_reduce_kernel<EPI>, dim3(blocks_for(total, 256, 4096u)), dim3(256), 0,
                       s, partial, splits, C, ldc, M, N, R, ldr);
    FMLH_LAUNCHED("splitk_reduce_kernel");
    return FMLH_OK;
}

int reduce_dispatch(int epi, const float* partial, int splits, float* C, int ldc, int M, int N,
                    const float* R, int ldr, hipStream_t s) {
    switch (epi) {
        case kEpiGelu: return launch_reduce<kEpiGelu>(partial, splits, C, ldc, M, N, R, ldr, s);
        case kEpiResid: return launch_reduce<kEpiResid>(partial, splits, C, ldc, M, N, R, ldr, s);
        default: return launch_reduce<kEpiNone>(partial, splits, C, ldc, M, N, R, ldr, s);
    }
}

template <int BM, int BN, bool BT, int EPI>
int launch_mfma(const GemmArgs& g, int splits, int k_per_split, float* ws) {
    dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, splits);
    if (splits > 1) {
        hipLaunchKernelGGL((gemm_mfma_kernel<BM, BN, BT, EPI, true>), grid, dim3(256), 0, g.s, g.A,
                           g.lda, g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr, ws, k_per_split);
        FMLH_LAUNCHED("gemm_mfma_kernel(split)");
        return reduce_dispatch(g.epi, ws, splits, g.C, g.ldc, g.M, g.N, g.R, g.ldr, g.s);
    }
    hipLaunchKernelGGL((gemm_mfma_kernel<BM, BN, BT, EPI, false>), grid, dim3(256), 0, g.s, g.A,
                       g.lda, g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr, nullptr, 0);
    FMLH_LAUNCHED("gemm_mfma_kernel");
    return FMLH_OK;
}

template <int BM, int BN, bool BT>
int mfma_epi(const GemmArgs& g, int splits, int kps, float* ws) {
    switch (g.epi) {
        case kEpiGelu: return launch_mfma<BM, BN, BT, kEpiGelu>(g, splits, kps, ws);
        case kEpiResid: return launch_mfma<BM, BN, BT, kEpiResid>(g, splits, kps, ws);
        default: return launch_mfma<BM, BN, BT, kEpiNone>(g, splits, kps, ws);
    }
}

template <int BM, int BN>
int mfma_tile(const GemmArgs& g, int splits, int kps, float* ws) {
    return g.b_trans ? mfma_epi<BM, BN, true>(g, splits, kps, ws)
                     : mfma_epi<BM, BN, false>(g, splits, kps, ws);
}

SplitGemm split_args(const GemmArgs& g, int tile) {
    SplitGemm q;
    q.A = g.A; q.lda = g.lda; q.B = g.B; q.ldb = g.ldb; q.b_kc = g.b_trans != 0;
    q.C = g.C; q.ldc = g.ldc; q.M = g.M; q.N = g.N; q.K = g.K; q.epi = g.epi; q.R = g.R; q.ldr = g.ldr;
    q.kv = g.kv; q.tile = tile; q.s = g.s;
    return q;
}

// A planned split product: one launch, or K ranges and their reduction with the epilogue.
int run_split(const GemmArgs& g, const GemmPlan& p, float* ws) {
    SplitGemm q = split_args(g, p.bm);
    q.k_groups = p.k_groups;
    if (p.splits == 1) return gemm_split(q);
    q.epi = kEpiNone; q.splits = p.splits; q.k_per_split = p.k_per_split; q.partial = ws;
    FMLH_TRY(gemm_split(q));
    return reduce_dispatch(g.epi, ws, p.splits, g.C, g.ldc, g.M, g.N, g.R, g.ldr, g.s);
}

template <int EPI>
int launch_nt(const GemmArgs& g) {
    const char* env = std::getenv("FMLH_GEMM_SKINNY");  // "quad": 16 lanes per column
    if (g.ln_g != nullptr || !(env && std::strcmp(env, "quad") == 0)) {
        // Waves per column so that the launch has >= ~2048 waves when N is small.
        const int ks = g.N <= 1024 ? 4 : (g.N <= 4096 ? 2 : 1);
        const char* wide = std::getenv("FMLH_SKINNY_WIDE_NC");  // columns per wave, N > 4096
        const int wnc = wide ? std::atoi(wide) : 4;
        if (ks == 1 && g.ln_g == nullptr && (wnc == 2 || wnc == 4)) {
            const unsigned wwgs = (unsigned)((g.N + 4 * wnc - 1) / (4 * wnc));
            if (wnc == 4)
                hipLaunchKernelGGL((skinny_nt_wide_kernel<EPI, 4>), dim3(wwgs), dim3(256), 0, g.s, g.A, g.lda,
                                   g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr);
            else
                hipLaunchKernelGGL((skinny_nt_wide_kernel<EPI, 2>), dim3(wwgs), dim3(256), 0, g.s, g.A, g.lda,
                                   g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr);
            FMLH_LAUNCHED("skinny_nt_wide_kernel");
            return FMLH_OK;
        }
        const unsigned wgs = (unsigned)((g.N * ks + 3) / 4);
#define FMLH_SKW(KSV, LNV)                                                                        \
    hipLaunchKernelGGL((skinny_nt_wave_kernel<EPI, KSV, LNV>), dim3(wgs), dim3(256), 0, g.s, g.A, g.lda, \
                       g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr, g.ln_g, g.ln_b, g.ln_eps)
        if (g.ln_g != nullptr) {
            if (ks == 4) FMLH_SKW(4, true);
            else if (ks == 2) FMLH_SKW(2, true);
            else FMLH_SKW(1, true);
        } else {
            if (ks == 4) FMLH_SKW(4, false);
            else if (ks == 2) FMLH_SKW(2, false);
            else FMLH_SKW(1, false);
        }
#undef FMLH_SKW
        FMLH_LAUNCHED("skinny_nt_wave_kernel");
        return FMLH_OK;
    }
    hipLaunchKernelGGL(skinny_nt_kernel<EPI>, dim3((g.N + 3) / 4), dim3(64), 0, g.s, g.A, g.lda,
                       g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, g.R, g.ldr);
    FMLH_LAUNCHED("skinny_nt_kernel");
    return FMLH_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The split-K NT kernel takes B stored N x K, 64 x 64 tiles and K ranges of at most
// kNtSplitMaxBlocks blocks (the callers have checked alignment and K % 16).
bool nt_split_applies(const GemmArgs& g, const GemmPlan& p) {
    const char* env = std::getenv("FMLH_GEMM_NT_SPLIT");  // "0": register-staged split kernel
    if (env && env[0] == '0') return false;
    return g.b_trans && p.kind == GemmPlan::kMfma && p.splits > 1 && p.bm == 64 && p.bn == 64 &&
           p.k_per_split % KB == 0 && p.k_per_split / KB <= kNtSplitMaxBlocks;
}

int launch_nt_split(const GemmArgs& g, const GemmPlan& p, float* ws) {
    dim3 grid((g.N + 63) / 64, (g.M + 63) / 64, p.splits);
    const size_t lds = (size_t)(p.k_per_split / KB) * 128 * KB * sizeof(float);
    hipLaunchKernelGGL(gemm_nt_split_kernel, grid, dim3(256), lds, g.s, g.A, g.lda, g.B, g.ldb, g.M,
                       g.N, p.k_per_split, ws);
    FMLH_LAUNCHED("gemm_nt_split_kernel");
    return FMLH_OK;
}

}  // namespace

// CUs to plan for (no device, as in the host-only tests of the plans: an MI355X's).
static int plan_cus() { return cu_count() > 0 ? cu_count() : 256; }

// Groups of waves per 64 x 64 tile: two where the launch has at most a work-group per CU and each
// at least four K blocks.
static int split_k_groups(float work_groups, int k) { return work_groups <= (float)plan_cus() && k >= 128 ? 2 : 1; }

GemmPlan plan_gemm(int M, int N, int K, int b_trans, bool one_range, size_t ws_max, bool split_takes) {
    GemmPlan p;
    if (M <= SK_MAXM) {
        if (b_trans) {
            p.kind = GemmPlan::kSkinnyNT;
        } else {
            p.kind = GemmPlan::kSkinnyNN;
            p.splits = (K + SK_KCHUNK - 1) / SK_KCHUNK;
            p.ws_elems = (size_t)p.splits * M * N;
        }
        return p;
    }
    const int cus = plan_cus();
    const long tiles64 = (long)((M + 63) / 64) * ((N + 63) / 64);
    const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    // Split bf16 tiles for everything wider than the batched decode, but for the smallest products,
    // which the fp32 MFMA kernels' K ranges spread over more CUs or which are over before the
    // split tiles' longer start is (us, fp32 / split): N x K weights of up to 36 tiles and K 768 on
    // gemm_nt_split_kernel (256 x 384 x 384 8.2 / 9.1; 256 x 1152 x 384 11.4 / 9.2), K x N ones up
    // to K 384 (256 x 384 x 384 9.3 / 9.7; 150 x 1024 x 256 8.6 / 8.1), and tiles times K to 4096
    // (1000 x 256 x 64 4.6 / 5.3).
    const bool small = (tiles64 <= 36 && K <= (b_trans ? 768 : 384)) || tiles64 * K <= 4096;
    if (split_takes && ((M > 64 && !small) || (b_trans && 2 * tiles64 >= cus))) {
        p.kind = GemmPlan::kSplit;
        // Tile and K ranges by the time (us) they take, fitted on MI355X to 266 shapes (256 .. 14336
        // rows of 384 .. 1024-wide blocks, K to 50304) x 2 layouts x up to 15 choices: 1 % behind the
        // best choice on average, 12 % at worst.  A CU multiplies a 128 x 128 x 16 block in 0.62 us
        // whether it holds one work-group or two, a 64 x 64 x 32 one in 0.64 alone (0.70 with B stored
        // K x N), 0.45 (0.50) by two groups of waves that share the K range, and 0.41 among several
        // work-groups; K ranges write and read their partials, and the reduction is a launch.  What
        // is left of the last work-group per CU counts half (large tiles: the CUs that have none
        // leave the others clock and bandwidth) or nearly whole (small ones); without that, 2048 x
        // 768 x 3072 took 92 us instead of 68, 2500 x 1024 x 4096 163 instead of 126.  Two groups
        // serve products of at most a tile per CU, whose one wave per SIMD would wait out every
        // latency (256 x 1536 x 384 11.1 -> 9.1, 1024 x 768 x 768 19.5 -> 14.3).
        float best = INFINITY;
        const float mn = (float)M * N;
        for (int tile : {128, 64}) {
            if (tile == 128 && tiles64 < cus / 2) continue;  // too few large tiles for the device
            const float tiles = (float)(tile == 128 ? tiles128 : tiles64), cu = (float)cus;
            const float block = tile == 128 ? (b_trans ? 0.62f / 16 : 0.665f / 16) : (b_trans ? 0.64f / 32 : 0.70f / 32);
            const float last = tile == 128 ? 0.5f : 0.85f;
            for (int sp : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64}) {
                // K ranges pay while CUs are idle, more than 16 while there is a CU for each and they stay
                // long (128 x 64 x 65536: 66 us in 16, 40 in 64, on the fp32 tiles' 64 ranges 52).
                if (sp > 1 && (one_range || tiles * (sp - 1) >= 3 * cu || K < 64 * sp || sp * mn > ws_max)) break;
                if (sp > 16 && (tiles * sp > cu || K < 512 * sp)) break;
                const float wgs = tiles * sp, kr = (float)K / sp;
                const float units = (1.0f - last) * wgs / cu + last * std::ceil(wgs / cu);
                const bool two = tile == 64 && split_k_groups(wgs, (int)kr) == 2;
                const float t = (tile == 128 ? std::max(1.0f, units) * block
                                 : two       ? 0.71f * block
                                             : std::max(block, units * (0.407f / 32))) * kr +
                                (sp > 1 ? 4.3f + 0.11f * sp + 0.12f * std::max(0, sp - 16) + 1.53e-6f * sp * mn : 1.08e-6f * mn);
                if (t < best) {
                    best = t;
                    p.bm = p.bn = tile;
                    p.splits = sp;
                    p.k_groups = two ? 2 : 1;
                }
            }
        }
        // FMLH_GEMM_NT_TILE=128x128 | 64x64 forces the tile, FMLH_GEMM_NT_SPLIT_K=n the K ranges
        // (0: one).
        if (const char* e = std::getenv("FMLH_GEMM_NT_TILE")) {
            int bm = 0, bn = 0;
            if (std::sscanf(e, "%dx%d", &bm, &bn) == 2 && (bm == 128 || bm == 64)) {
                p.bm = p.bn = bm;
                p.k_groups = bm == 64 ? split_k_groups((float)tiles64 * p.splits, K / p.splits) : 1;
            }
        }
        if (const char* e = one_range ? nullptr : std::getenv("FMLH_GEMM_NT_SPLIT_K")) p.splits = std::max(1, std::atoi(e));
        if (p.splits > 1) {
            const int kb = p.bm == 64 ? 32 : 16;  // whole K blocks of the tile
            p.k_per_split = ((K + p.splits - 1) / p.splits + kb - 1) / kb * kb;
            p.splits = (K + p.k_per_split - 1) / p.k_per_split;
            p.ws_elems = p.splits > 1 ? (size_t)p.splits * M * N : 0;
        }
        return p;
    }
    p.kind = GemmPlan::kMfma;
    const long t128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64);
    long tiles;
    if (t128 >= cus) { p.bm = 128; p.bn = 128; tiles = t128; }
    else { p.bm = 64; p.bn = 64; tiles = t64; }
    // Split K when the tile grid cannot fill the device (skinny batched-decode shapes).
    int splits = 1;
    while (tiles * splits * 2 <= cus && K / (splits * 2) >= 64 && (K / (splits * 2)) % KB == 0)
        splits *= 2;
    p.splits = splits;
    p.k_per_split = K / splits;
    p.ws_elems = splits > 1 ? (size_t)splits * M * N : 0;
    return p;
}

namespace {
// The plan of a call: that of plan_rows rows where given, with room for the call's own.  Row strides
// beyond the split tiles' 32-bit offsets stay on the fp32 MFMA tiles.
GemmPlan plan_for(const GemmArgs& g) {
    GemmPlan p = plan_gemm(std::max(g.M, g.plan_rows), g.N, g.K, g.b_trans, g.epi == kEpiKV, g.ws_max,
                           gemm_split_takes(split_args(g, 64)));
    if (g.plan_rows > g.M && p.splits > 1) p.ws_elems = (size_t)p.splits * g.M * g.N;
    return p;
}
}  // namespace

bool gemm_takes_ln(int M, int N, int K, int b_trans) {
    return M > 0 && N > 0 && K <= 64 * kSkLnNE && plan_gemm(M, N, K, b_trans).kind == GemmPlan::kSkinnyNT;
}

bool gemm_runs_nt(const GemmArgs& g) {
    const bool vec_ok = aligned16(g.A) && aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                        g.K % KB == 0;
    return vec_ok && g.M > 0 && g.N > 0 && g.b_trans && plan_for(g).kind == GemmPlan::kSplit;
}

size_t engine_workspace_elems(int C, int V, int batch, int rows) {
    const int M = batch * rows;
    return std::max({plan_gemm(M, 3 * C, C, 1).ws_elems, plan_gemm(M, C, C, 1).ws_elems, plan_gemm(M, 4 * C, C, 1).ws_elems,
                     plan_gemm(M, C, 4 * C, 1).ws_elems, plan_gemm(batch, V, C, 1).ws_elems});
}

size_t gemm_workspace_elems(const GemmArgs& g) {
    if (g.M == 0 || g.N == 0 || g.K == 0) return 0;
    const bool vec_ok = aligned16(g.A) && aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                        g.K % KB == 0;
    return vec_ok ? plan_for(g).ws_elems : 0;  // the strided fallback takes none
}

int gemm(const GemmArgs& g, float* ws, size_t ws_elems) {
    if (g.M == 0 || g.N == 0) return FMLH_OK;
    FMLH_REQUIRE(g.K > 0, "gemm: K == 0");
    FMLH_REQUIRE(g.ln_g == nullptr || gemm_takes_ln(g.M, g.N, g.K, g.b_trans),
                 "gemm: a LayerNorm on A needs the skinny NT path (M <= 8, K <= 1024)");
    FMLH_REQUIRE(g.epi != kEpiKV || (gemm_runs_nt(g) && g.kv.kc && g.kv.vc && g.N == 3 * g.kv.C &&
                                     g.kv.hd > 0 && (g.kv.hd & (g.kv.hd - 1)) == 0),
                 "gemm: the cache-writing epilogue needs the NT kernel, N = 3 C and a power-of-two head_dim");
    const bool vec_ok = aligned16(g.A) && aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                        g.K % KB == 0;
    FMLH_REQUIRE(g.ln_g == nullptr || (vec_ok && aligned16(g.ln_g) && (g.ln_b == nullptr || aligned16(g.ln_b))),
                 "gemm: a LayerNorm on A needs 16-byte aligned rows and parameters");
    if (!vec_ok) {
        // Fallback: generic strided kernel, then the epilogue through the reduce kernel.
        FMLH_REQUIRE(g.epi == kEpiNone, "gemm: epilogue needs 16-byte aligned rows with K %% 16 == 0");
        return gemm_strided(g.b_trans ? FMLH_TRANSPOSE_RIGHT : FMLH_TRANSPOSE_NONE, g.C, g.A, g.B,
                            g.M, g.N, g.K, g.lda, 1, g.ldb, 1, g.ldc, 1, 1, 0, 0, 0, g.s);
    }
    GemmPlan p = plan_for(g);
    if (p.ws_elems > ws_elems) {
        if (ws != nullptr) return set_error(FMLH_E_INVALID, "gemm: workspace too small");
        const int rc = global_workspace(p.ws_elems, &ws);
        if (rc != FMLH_OK && p.kind != GemmPlan::kSplit) return rc;
        if (rc != FMLH_OK) {  // no room for partials: one K range
            (void)hipGetLastError();
            clear_error();
            p.splits = 1;
        }
    }
    switch (p.kind) {
        case GemmPlan::kSkinnyNT:
            switch (g.epi) {
                case kEpiGelu: return launch_nt<kEpiGelu>(g);
                case kEpiResid: return launch_nt<kEpiResid>(g);
                default: return launch_nt<kEpiNone>(g);
            }
        case GemmPlan::kSkinnyNN: {
            dim3 grid((g.N + 255) / 256, p.splits);
            hipLaunchKernelGGL(skinny_nn_partial_kernel, grid, dim3(64), 0, g.s, g.A, g.lda, g.B,
                               g.ldb, ws, g.M, g.N, g.K);
            FMLH_LAUNCHED("skinny_nn_partial_kernel");
            return reduce_dispatch(g.epi, ws, p.splits, g.C, g.ldc, g.M, g.N, g.R, g.ldr, g.s);
        }
        case GemmPlan::kSplit: return run_split(g, p, ws);
        default:
            if (nt_split_applies(g, p)) {
                FMLH_TRY(launch_nt_split(g, p, ws));
                return reduce_dispatch(g.epi, ws, p.splits, g.C, g.ldc, g.M, g.N, g.R, g.ldr, g.s);
            }
            if (p.bm == 128) return mfma_tile<128, 128>(g, p.splits, p.k_per_split, ws);
            return mfma_tile<64, 64>(g, p.splits, p.k_per_split, ws);
    }
}

int gemm_nt_partials(const GemmArgs& g, int splits, float* ws, size_t ws_elems) {
    const bool vec_ok = aligned16(g.A) && aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0;
    FMLH_REQUIRE(g.b_trans && vec_ok && splits >= 1 && g.K % (splits * KB) == 0,
                 "gemm_nt_partials: %dx%dx%d in %d splits needs B stored N x K, 16-byte rows, K %% (16 splits) == 0",
                 g.M, g.N, g.K, splits);
    FMLH_REQUIRE(ws != nullptr && (size_t)splits * g.M * g.N <= ws_elems, "gemm_nt_partials: workspace too small");
    if (g.M == 0 || g.N == 0) return FMLH_OK;
    SplitGemm q = split_args(g, 64);
    q.epi = kEpiNone; q.splits = splits; q.k_per_split = g.K / splits; q.partial = ws;
    q.k_groups = split_k_groups((float)((std::max(g.M, g.plan_rows) + 63) / 64) * ((g.N + 63) / 64) * splits, q.k_per_split);
    if (splits == 1) { q.C = ws; q.ldc = g.N; }
    return gemm_split(q);
}

int gemm_split_partials(const GemmArgs& g, float* ws, size_t ws_elems, int* splits) {
    *splits = 0;
    const bool vec_ok = aligned16(g.A) && aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                        g.K % KB == 0;
    if (g.M == 0 || g.N == 0 || !vec_ok) return FMLH_OK;
    const GemmPlan p = plan_gemm(g.M, g.N, g.K, g.b_trans);
    if (p.kind != GemmPlan::kMfma || p.splits < 2) return FMLH_OK;
    FMLH_REQUIRE(ws != nullptr && p.ws_elems <= ws_elems, "gemm_split_partials: workspace too small");
    if (nt_split_applies(g, p)) {
        *splits = p.splits;
        return launch_nt_split(g, p, ws);
    }
    dim3 grid((g.N + p.bn - 1) / p.bn, (g.M + p.bm - 1) / p.bm, p.splits);
#define FMLH_PARTIALS(BMV, BTV)                                                                  \
    hipLaunchKernelGGL((gemm_mfma_kernel<BMV, BMV, BTV, kEpiNone, true>), grid, dim3(256), 0, g.s, \
                       g.A, g.lda, g.B, g.ldb, g.C, g.ldc, g.M, g.N, g.K, nullptr, 0, ws, p.k_per_split)
    if (p.bm == 128) {
        if (g.b_trans) FMLH_PARTIALS(128, true); else FMLH_PARTIALS(128, false);
    } else {
        if (g.b_trans) FMLH_PARTIALS(64, true); else FMLH_PARTIALS(64, false);
    }
#undef FMLH_PARTIALS
    FMLH_LAUNCHED("gemm_mfma_kernel(split partials)");
    *splits = p.splits;
    return FMLH_OK;
}

namespace {
// Whether a strided product runs on the split bf16 tiles; fills everything but the output.  They
// take views with a contiguous index on either side from 64 tiles' worth of outputs on: fewer
// leave CUs idle that the wave-split kernel's 16 x 16 tiles still use (us, that kernel / this one:
// 24 tiles 256 x 64 x 256 6.1 / 9.1, 16 tiles 256 x 256 x 2048 20 / 48; 64 tiles 512 x 64 x 512 19
// / 14.8; 192 tiles 1024 x 64 x 1024 41 / 26; 576 tiles 3072 x 768 x 1024 96 / 49).  The error is below
// that of that kernel's four K ranges (K 1024: 2.9e-7 / 1.9e-7).  128 x 128 tiles from two per CU on
// (1024 x 1024 x 64, 12 planes: 27.0 / 28.0) where they compute at most a quarter more than 64 x 64
// ones (1024 planes of 16 x 64 x 256: 51 us in large tiles, 21 in small ones; 64 x 64 x 256 47, 28).
bool strided_split(bool tl, bool tr, const float* L, const float* R, uint32_t M, uint32_t N, uint32_t K, uint32_t l_rs,
                   uint32_t l_cs, uint32_t r_rs, uint32_t r_cs, uint32_t o_rs, uint32_t o_cs, uint32_t batch,
                   size_t l_plane, size_t r_plane, SplitGemm* q) {
    if (o_cs != 1 || o_rs > INT32_MAX || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || batch > 65535) return false;
    if ((double)M * N * batch < 64.0 * 64 * 64) return false;
    // Planes of a quarter tile beyond one per CU stay on that kernel's 32 x 32 tiles but for the shortest
    // K (32 x 32 x 256: 256 planes 10 / 8.5 us, 400 10 / 12, 1024 x 32 x 32 x 64 7.1 / 9.5, 600 x 32 x 32 x 16 6 / 5.5).
    if (M <= 32 && N <= 32 && K > 32 && batch > (uint32_t)plan_cus()) return false;
    // Strides between the k of one row of A (column of B) and between its rows (columns).
    const uint32_t a_k = tl ? l_rs : l_cs, a_r = tl ? l_cs : l_rs, b_k = tr ? r_cs : r_rs, b_r = tr ? r_rs : r_cs;
    if ((a_k != 1 && a_r != 1) || (b_k != 1 && b_r != 1)) return false;
    q->A = L; q->a_kc = a_k == 1; q->lda = (int)std::min<uint32_t>(a_k == 1 ? a_r : a_k, INT32_MAX); q->a_plane = l_plane;
    q->B = R; q->b_kc = b_k == 1; q->ldb = (int)std::min<uint32_t>(b_k == 1 ? b_r : b_k, INT32_MAX); q->b_plane = r_plane;
    q->M = (int)M; q->N = (int)N; q->K = (int)K; q->planes = (int)batch;
    const uint64_t tiles = (uint64_t)((M + 63) / 64) * ((N + 63) / 64) * batch;
    const uint64_t large = (uint64_t)((M + 127) / 128) * ((N + 127) / 128) * batch;
    q->tile = large >= 2u * plan_cus() && 16 * large <= 5 * tiles ? 128 : 64;
    if (q->tile == 64) q->k_groups = split_k_groups((float)tiles, (int)K);
    return gemm_split_takes(*q);
}
}  // namespace

int gemm_strided(int mode, float* out, const float* L, const float* R, uint32_t M, uint32_t N,
                 uint32_t K, uint32_t l_rs, uint32_t l_cs, uint32_t r_rs, uint32_t r_cs,
                 uint32_t o_rs, uint32_t o_cs, uint32_t batch, size_t l_plane, size_t r_plane,
                 size_t o_plane, hipStream_t s) {
    if (M == 0 || N == 0 || batch == 0) return FMLH_OK;
    const bool tl = mode == FMLH_TRANSPOSE_LEFT || mode == FMLH_TRANSPOSE_BOTH;
    const bool tr = mode == FMLH_TRANSPOSE_RIGHT || mode == FMLH_TRANSPOSE_BOTH;
    {
        SplitGemm q;
        if (strided_split(tl, tr, L, R, M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, batch, l_plane, r_plane, &q)) {
            q.C = out; q.ldc = (int)o_rs; q.c_plane = o_plane; q.s = s;
            return gemm_split(q);
        }
    }
    // K within one 64-wide chunk: one chunk per 32 x 32 tile.  Longer K: the wave-split
    // kernel, with 16 x 16 tiles unless 32 x 32 tiles already give a work-group per CU.
    const size_t tiles32 = (size_t)((N + 31) / 32) * ((M + 31) / 32) * batch;
    const int kind = K <= kStKC || std::getenv("FMLH_STRIDED_NO_WSPLIT") ? 0 : (tiles32 >= (size_t)cu_count() ? 32 : 16);
    const uint32_t tt = kind == 16 ? 16u : 32u;
    dim3 grid((N + tt - 1) / tt, (M + tt - 1) / tt, batch);
#define FMLH_STRIDED(TLV, TRV)                                                                             \
    do {                                                                                                    \
        if (kind == 16)                                                                                     \
            hipLaunchKernelGGL((gemm_strided_wsplit_kernel<TLV, TRV, 16>), grid, dim3(256), 0, s, out, L, R,  \
                               M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, l_plane, r_plane, o_plane);       \
        else if (kind == 32)                                                                                \
            hipLaunchKernelGGL((gemm_strided_wsplit_kernel<TLV, TRV, 32>), grid, dim3(256), 0, s, out, L, R,  \
                               M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, l_plane, r_plane, o_plane);       \
        else                                                                                                \
            hipLaunchKernelGGL((gemm_strided_kernel<TLV, TRV>), grid, dim3(256), 0, s, out, L, R, M, N, K,    \
                               l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, l_plane, r_plane, o_plane);               \
    } while (0)
    if (tl && tr) FMLH_STRIDED(true, true);
    else if (tl) FMLH_STRIDED(true, false);
    else if (tr) FMLH_STRIDED(false, true);
    else FMLH_STRIDED(false, false);
#undef FMLH_STRIDED
    FMLH_LAUNCHED("gemm_strided_kernel");
    return FMLH_OK;
}

}  // namespace fmlh

using namespace fmlh;

extern "C" {

int fmlh_mul(int mode, float* out, const float* L, const float* R, uint32_t M, uint32_t N,
             uint32_t K) {
    FMLH_REQUIRE(out && L && R, "fmlh_mul: null pointer");
    FMLH_REQUIRE(mode >= 0 && mode <= 3, "fmlh_mul: bad transpose mode %d", mode);
    FMLH_TRY(ensure_init());
    if (mode == FMLH_TRANSPOSE_NONE || mode == FMLH_TRANSPOSE_RIGHT) {
        GemmArgs g;
        g.A = L; g.lda = (int)K;
        g.B = R; g.ldb = (int)(mode == FMLH_TRANSPOSE_RIGHT ? K : N);
        g.b_trans = mode == FMLH_TRANSPOSE_RIGHT;
        g.C = out; g.ldc = (int)N;
        g.M = (int)M; g.N = (int)N; g.K = (int)K;
        g.s = stream();
        return gemm(g, nullptr, 0);
    }
    const bool tl = true;
    const bool tr = mode == FMLH_TRANSPOSE_BOTH;
    return gemm_strided(mode, out, L, R, M, N, K, tl ? M : K, 1, tr ? K : N, 1, N, 1, 1, 0, 0, 0,
                        stream());
}

int fmlh_gemm_ex(const float* A, int lda, const float* B, int ldb, int b_trans, float* C, int ldc,
                 int M, int N, int K, int epilogue, const float* R, int ldr) {
    FMLH_REQUIRE(A && B && C, "fmlh_gemm_ex: null pointer");
    FMLH_REQUIRE(M >= 0 && N >= 0 && K >= 0, "fmlh_gemm_ex: negative size");
    FMLH_REQUIRE(epilogue >= kEpiNone && epilogue <= kEpiResid, "fmlh_gemm_ex: bad epilogue %d",
                 epilogue);
    FMLH_REQUIRE(epilogue != kEpiResid || R != nullptr, "fmlh_gemm_ex: residual needs R");
    FMLH_REQUIRE(lda >= K && ldc >= N && ldb >= (b_trans ? K : N), "fmlh_gemm_ex: bad leading dim");
    FMLH_TRY(ensure_init());
    GemmArgs g;
    g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.b_trans = b_trans ? 1 : 0;
    g.C = C; g.ldc = ldc; g.M = M; g.N = N; g.K = K; g.epi = epilogue; g.R = R; g.ldr = ldr;
    g.ws_max = kNoAllocScratchFloats;  // the plan of fmlh_gemm_ex_noalloc, whose results are the same
    g.s = stream();
    return gemm(g, nullptr, 0);
}

int fmlh_gemm_ex_noalloc(const float* A, int lda, const float* B, int ldb, int b_trans, float* C, int ldc,
                         int M, int N, int K, int epilogue, const float* R, int ldr) {
    FMLH_REQUIRE(A && B && C, "fmlh_gemm_ex_noalloc: null pointer");
    FMLH_REQUIRE(M >= 0 && N >= 0 && K >= 0, "fmlh_gemm_ex_noalloc: negative size");
    FMLH_REQUIRE(epilogue >= kEpiNone && epilogue <= kEpiResid, "fmlh_gemm_ex_noalloc: bad epilogue %d",
                 epilogue);
    FMLH_REQUIRE(epilogue != kEpiResid || R != nullptr, "fmlh_gemm_ex_noalloc: residual needs R");
    FMLH_REQUIRE(lda >= K && ldc >= N && ldb >= (b_trans ? K : N), "fmlh_gemm_ex_noalloc: bad leading dim");
    // No lazy initialisation here (it would create the library stream): fmlh_init set up the
    // scratch address of this device.
    float* ws = noalloc_scratch();
    if (ws == nullptr)
        return set_error(FMLH_E_STATE, "fmlh_gemm_ex_noalloc: call fmlh_init first (it sets up the scratch)");
    GemmArgs g;
    g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.b_trans = b_trans ? 1 : 0;
    g.C = C; g.ldc = ldc; g.M = M; g.N = N; g.K = K; g.epi = epilogue; g.R = R; g.ldr = ldr;
    g.ws_max = kNoAllocScratchFloats;
    g.s = stream();
    const size_t need = gemm_workspace_elems(g);
    if (need > kNoAllocScratchFloats)
        return set_error(FMLH_E_INVALID,
                         "fmlh_gemm_ex_noalloc: %dx%dx%d needs %zu floats of split-K partials; the fixed "
                         "scratch holds %zu (use fmlh_gemm_ex)", M, N, K, need, kNoAllocScratchFloats);
    return gemm(g, ws, kNoAllocScratchFloats);
}

int fmlh_matmul_strided(int mode, float* out, const float* L, const float* R, uint32_t M,
                        uint32_t N, uint32_t K, uint32_t l_rs, uint32_t l_cs, uint32_t r_rs,
                        uint32_t r_cs, uint32_t o_rs, uint32_t o_cs, uint32_t batch,
                        size_t l_plane, size_t r_plane, size_t o_plane) {
    FMLH_REQUIRE(out && L && R, "fmlh_matmul_strided: null pointer");
    FMLH_REQUIRE(mode >= 0 && mode <= 3, "fmlh_matmul_strided: bad transpose mode %d", mode);
    FMLH_TRY(ensure_init());
    return gemm_strided(mode, out, L, R, M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, batch,
                        l_plane, r_plane, o_plane, stream());
}

}  // extern "C"

namespace fmlh {

// ---- split-K partials of fmlh_gemm_ex_noalloc ------------------------------------------------
// A fixed device array, one copy per device (each device that loads the library holds it until
// the process ends).  In host code `scratch` names a host-side stand-in, not device memory: the
// device address comes from hipGetSymbolAddress, once per device, at fmlh_init.

static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};
int g_scratch_device = -1;  // the device the library runs on (fmlh_init)
}  // namespace

int setup_noalloc_scratch(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0 || device >= kMaxDevices)
        return set_error(FMLH_E_INVALID, "device %d beyond the %d the scratch table holds", device, kMaxDevices);
    if (g_scratch_ptr[device] == nullptr) {
        void* p = nullptr;
        FMLH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[device] = static_cast<float*>(p);
    }
    g_scratch_device = device;
    return FMLH_OK;
}

float* noalloc_scratch() {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (stream() == nullptr || g_scratch_device < 0) return nullptr;  // not initialised
    return g_scratch_ptr[g_scratch_device];
}

// ---- plans, for tests (no device needed) ----------------------------------------------------

extern "C" int fmlh_internal_plan(int M, int N, int K, int b_trans, int lda, int ldb, int* kind, int* tile, int* k_groups,
                                  int* splits, size_t* ws_elems) {
    GemmArgs g;
    g.M = M; g.N = N; g.K = K; g.b_trans = b_trans; g.lda = lda; g.ldb = ldb;
    const GemmPlan p = plan_for(g);
    *kind = p.kind; *tile = p.bm; *k_groups = p.k_groups; *splits = p.splits; *ws_elems = p.ws_elems;
    return FMLH_OK;
}

extern "C" int fmlh_internal_strided_tile(int mode, uint32_t M, uint32_t N, uint32_t K, uint32_t l_rs, uint32_t l_cs,
                                          uint32_t r_rs, uint32_t r_cs, uint32_t o_rs, uint32_t o_cs, uint32_t batch,
                                          size_t l_plane, size_t r_plane) {
    SplitGemm q;
    const bool tl = mode == FMLH_TRANSPOSE_LEFT || mode == FMLH_TRANSPOSE_BOTH;
    const bool tr = mode == FMLH_TRANSPOSE_RIGHT || mode == FMLH_TRANSPOSE_BOTH;
    return strided_split(tl, tr, nullptr, nullptr, M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, batch, l_plane, r_plane, &q)
               ? q.tile : 0;
}

extern "C" size_t fmlh_internal_engine_workspace(int C, int V, int batch, int rows) {
    return engine_workspace_elems(C, V, batch, rows);
}

void release_global_workspace() {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    if (g_ws) (void)hipFree(g_ws);
    g_ws = nullptr;
    g_ws_elems = 0;
}

}  // namespace fmlh

// fp32 products on the bf16 matrix cores: gemm_split_kernel.
//
// Every fp32 operand element is split exactly into three bf16 parts, x = x0 + x1 + x2 (each the
// round-to-nearest bf16 of what is left, 3 x 8 significant bits = fp32's 24; the method of Henry, Tang
// and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019), and the product
// takes the six part products whose weight is 2^-16 or more of the whole,
//   a b ~ a0 b0 + (a0 b1 + a1 b0) + (a0 b2 + a1 b1 + a2 b0),
// accumulated in fp32 by the bf16 MFMAs: a0 b0 in one accumulator, the five small ones, smallest
// first, in another that is added at the end.  (In one accumulator each of the six MFMAs rounds the
// whole sum, and those roundings are not quite unbiased: 2-norm error 4.2e-7 instead of 1.6e-7 at K
// = 768, and a long decode after a prefill came out less exact than on fp32 MFMAs, 4.1e-7 / 2.8e-7.)
// The three products left out are below 2^-24 of |a b| together, under the rounding of one fp32
// product.
//
// Why: the fp32 MFMA these products ran on reaches 154 TFLOP/s at most on MI355X (100-113 of it
// in the kernel this one replaced); bf16 runs at 16 times its nominal rate, so six part products
// are 2.6 times as fast at the nominal peaks.  A large library bf16 product reaches 1218
// TFLOP/s, a sixth of which is 203: the 128 x 128 tiles reach 190 at 8192^3.  Measured, before ->
// after (us): 4096 x 3072 x 768 stored N x K 180 -> 107, 1024 x 50304 x 768 692 -> 452.  Relative
// error against 64 bits (2-norm, normal operands): K 384 / 768 / 3072 1.1e-7 / 1.6e-7 / 3.4e-7 (fp32
// MFMA: 3.5e-7 / 5.0e-7 / 9.9e-7).
//
// The operands are split while they are staged (registers -> LDS), so fp32 matrices of any
// layout are read once and nothing is kept.  Per 128 x 128 x 16 block a work-group's matrix cores
// need 768 clocks, its LDS 580 (three planes written once, read by two waves; 192 of them bank
// conflicts) and its vector units 600 (6 instructions per element and the addresses); per 64 x 64 x 32
// block, with half as many products per element, 384, 390 and 640 (counters).  The small tiles serve
// the products with too few large ones.  The
// launch bounds matter: left alone, the compiler takes 267 registers for the large tile (one wave
// per SIMD: 4096 x 3072 x 768 125 us instead of 107).
#include "bf16_split.h"
#include "gemm_split.h"

namespace fmlh {

namespace {

__device__ __forceinline__ float gelu_ref(float x) { return 0.5f * x * (1.0f + erff(x / 1.41421354f)); }

// Elements are staged times 2^24 and sums taken back by 2^-48, both exact.  bf16 numbers end at 2^-133
// (the MFMAs take subnormal ones as they are: measured), so unscaled, the parts of an element below
// 2^-110 no longer add up to it, which showed where it met the only large partner of its row.  Scaled,
// the parts of every fp32 number, subnormal ones included, are zero or normal.  Elements from
// 2^104 and sums from 2^80 on leave the range at its upper end instead and are multiplied again in
// fp32.  The multiplication costs 1 % (dense layers of a 768-wide block on 2500 rows 266 -> 270 us); flagging
// tiny elements instead, and testing sums against them, cost 2 to 3.5.
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// The MFMAs of the two tile sizes.  Lane l of an MT x MT product supplies row / column l % MT and
// the 8 consecutive k of octet l / MT; accumulator register r holds row 8 (r / 4) + 4 (l / MT) +
// r % 4 of column l % MT.
template <int MT>
struct Mfma;
template <>
struct Mfma<32> {
    using Acc = floatx16;
    static constexpr int kRegs = 16, kK = 16;
    static __device__ __forceinline__ Acc bf16(bf16x8 a, bf16x8 b, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ Acc fp32(float a, float b, Acc c) {  // one k per lane: l / MT
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mfma<16> {
    using Acc = floatx4;
    static constexpr int kRegs = 4, kK = 32;
    static __device__ __forceinline__ Acc bf16(bf16x8 a, bf16x8 b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ Acc fp32(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

template <int BM, int BN, int BK, int WVM, int WVN, int KG, bool AKC, bool BKC, int EPI, bool SPLIT, int MT>
__global__ __launch_bounds__(64 * WVM * WVN * KG, KG == 2 || BM == 128 ? 2 : 3) void gemm_split_kernel(
    const float* __restrict__ A, int lda, size_t a_plane, const float* __restrict__ B, int ldb, size_t b_plane,
    float* C, int ldc, size_t c_plane, int M, int N, int K, const float* R, int ldr, KvDest kv,
    float* __restrict__ partial, int k_per_split, int tiles_m, int tiles_n) {
    constexpr int U = BK / 8;                       // 16-byte units per row and plane
    constexpr int NT = 64 * WVM * WVN;
    constexpr int NA = BM * U / NT, NB = BN * U / NT;  // units a thread stages per K block
    static_assert(NA * NT == BM * U && NB * NT == BN * U, "units must divide over the threads");
    constexpr int WM = BM / WVM, WN = BN / WVN;
    constexpr int MB = WM / MT, NBK = WN / MT;     // MFMA tiles per wave
    using Acc = typename Mfma<MT>::Acc;
    constexpr int AR = Mfma<MT>::kRegs, KM = Mfma<MT>::kK;
    constexpr int STAGE = 3 * (BM + BN) * U;        // units per LDS stage
    extern __shared__ __attribute__((aligned(16))) uintx4 all_lds[];

    // KG = 2: two groups of waves, each with half of the K range and its own LDS stages.
    const int grp_k = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int tid = KG == 1 ? threadIdx.x : threadIdx.x % NT;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WVN, wn = wave % WVN;
    const int h = lane / MT, c = lane % MT;  // this lane's k octet and row / column of an MFMA

    // Tile order: consecutive work-groups go to different XCDs, so XCD x takes a contiguous
    // eighth of the tiles, walked in groups of 8 tile rows (their A rows and the walked B
    // columns stay in that XCD's L2).
    const int total = tiles_m * tiles_n;
    int t = blockIdx.x;
    {
        const int per = total / 8, rem = total % 8, x = t & 7, i = t >> 3;
        t = x * per + (x < rem ? x : rem) + i;
    }
    const int gsz = 8 * tiles_n, grp = t / gsz, gm = min(8, tiles_m - 8 * grp);
    const int tm = 8 * grp + (t - grp * gsz) % gm, tn = (t - grp * gsz) / gm;
    const int row0 = tm * BM, col0 = tn * BN;
    const int z = blockIdx.z;
    const int kbeg_wg = SPLIT ? z * k_per_split : 0;
    const int kend_wg = SPLIT ? min(K, kbeg_wg + k_per_split) : K;
    const int k_half = KG == 1 ? 0 : (max(kend_wg - kbeg_wg, 0) + 2 * BK - 1) / (2 * BK) * BK;
    const int kbeg = kbeg_wg + grp_k * k_half;
    const int kend = KG == 1 || grp_k ? kend_wg : min(kend_wg, kbeg_wg + k_half);
    uintx4* lds = all_lds + (size_t)grp_k * 2 * STAGE;
    if constexpr (!SPLIT) {
        A += z * a_plane;
        B += z * b_plane;
        C += z * c_plane;
    }

    // Staging: unit u = tid + 256 i of an operand is 8 consecutive k of one tile row.  K
    // contiguous: two 16-byte loads; row contiguous (stored K x rows): eight 4-byte loads,
    // consecutive lanes on consecutive rows.
    uint32_t a_off[NA], b_off[NB];  // bytes from the tile's base
    int a_row[NA], a_oct[NA], b_row[NB], b_oct[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int u = tid + NT * i;
        a_row[i] = AKC ? u / U : u % BM;
        a_oct[i] = AKC ? u % U : u / BM;
        const uint32_t r = min(a_row[i], M - 1 - row0);
        a_off[i] = 4u * (AKC ? r * (uint32_t)lda + 8 * a_oct[i] : 8 * a_oct[i] * (uint32_t)lda + r);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int u = tid + NT * i;
        b_row[i] = BKC ? u / U : u % BN;
        b_oct[i] = BKC ? u % U : u / BN;
        const uint32_t r = min(b_row[i], N - 1 - col0);
        b_off[i] = 4u * (BKC ? r * (uint32_t)ldb + 8 * b_oct[i] : 8 * b_oct[i] * (uint32_t)ldb + r);
    }
    const float* a_base = A + (AKC ? (size_t)row0 * lda : (size_t)row0);
    const float* b_base = B + (BKC ? (size_t)col0 * ldb : (size_t)col0);
    float va[NA][8], vb[NB][8];
    // (not full: element e of a unit at kk is zero from kend on, read at kend - 1; loads under a
    // condition would wait for one another)
    auto load_unit = [&](float (&v)[8], const float* base, uint32_t off, bool kc, int ld, int kk, bool full) {
        const char* p = reinterpret_cast<const char*>(base) + off;
        if (kc && (full || kend % 8 == 0)) {  // units are whole or past the end
            const char* q = full ? p : p + 4 * (min(kk, kend - 8) - kk);
            const floatx4 lo = *reinterpret_cast<const floatx4*>(q);
            const floatx4 hi = *reinterpret_cast<const floatx4*>(q + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = full || kk < kend ? lo[e] : 0.0f;
                v[4 + e] = full || kk < kend ? hi[e] : 0.0f;
            }
        } else if (full) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const float*>(p + (size_t)4 * e * ld);
        } else {
            const ptrdiff_t step = kc ? 4 : (ptrdiff_t)4 * ld;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = *reinterpret_cast<const float*>(p + (min(kk + e, kend - 1) - kk) * step);
                v[e] = kk + e < kend ? x : 0.0f;
            }
        }
    };
    auto load = [&](int k0, bool full) {
        const float* ab = a_base + (AKC ? (size_t)k0 : (size_t)k0 * lda);
        const float* bb = b_base + (BKC ? (size_t)k0 : (size_t)k0 * ldb);
#pragma unroll
        for (int i = 0; i < NA; ++i) load_unit(va[i], ab, a_off[i], AKC, lda, k0 + 8 * a_oct[i], full);
#pragma unroll
        for (int i = 0; i < NB; ++i) load_unit(vb[i], bb, b_off[i], BKC, ldb, k0 + 8 * b_oct[i], full);
    };
    // Unit o of row r is stored at o ^ swz(r): any 8 consecutive lanes, reading one row each or
    // writing, touch 8 distinct 16-byte bank groups.
    auto swz = [](int r) { return U == 2 ? (r >> 2) & 1 : (r >> 1) & 3; };
    auto store = [&](int st) {
        uintx4* sa = lds + st * STAGE;
        uintx4* sb = sa + 3 * BM * U;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            uintx4 p[3];
            split8(va[i], p, kSplitScale);
#pragma unroll
            for (int q = 0; q < 3; ++q) sa[(q * BM + a_row[i]) * U + (a_oct[i] ^ swz(a_row[i]))] = p[q];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            uintx4 p[3];
            split8(vb[i], p, kSplitScale);
#pragma unroll
            for (int q = 0; q < 3; ++q) sb[(q * BN + b_row[i]) * U + (b_oct[i] ^ swz(b_row[i]))] = p[q];
        }
    };

    Acc acc[MB][NBK], low[MB][NBK];  // a0 b0; the five small part products
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NBK; ++j)
#pragma unroll
                for (int r = 0; r < AR; ++r) acc[i][j][r] = 0.0f;
    };
    clear();
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NBK; ++j) low[i][j] = acc[i][j];

    // Two LDS stages, one barrier per K block: block k + 1 (in registers since the iteration
    // before) is split and written while block k is multiplied, block k + 2 is requested.  The
    // barrier waits for LDS only; the requested loads stay in flight across it.  Past the last
    // whole block the loop stages that block again (never multiplied), so its body has no branch
    // and the split's vector instructions run beside the MFMAs.
    auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto multiply = [&](int st, auto stage_next) {
        const uintx4* sa = lds + st * STAGE;
        const uintx4* sb = sa + 3 * BM * U;
#pragma unroll
        for (int ks = 0; ks < BK / KM; ++ks) {
            const int o = KM / 8 * ks + h;
            bf16x8 a[3][MB], b[3][NBK];
#pragma unroll
            for (int q = 2; q >= 0; --q) {
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    const int r = wm * WM + MT * i + c;
                    a[q][i] = __builtin_bit_cast(bf16x8, sa[(q * BM + r) * U + (o ^ swz(r))]);
                }
#pragma unroll
                for (int j = 0; j < NBK; ++j) {
                    const int r = wn * WN + MT * j + c;
                    b[2 - q][j] = __builtin_bit_cast(bf16x8, sb[((2 - q) * BN + r) * U + (o ^ swz(r))]);
                }
            }
            if (ks == 0) stage_next();
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NBK; ++j) {
                        Acc& d = q < 5 ? low[i][j] : acc[i][j];
                        d = Mfma<MT>::bf16(a[kSplitA[q]][i], b[kSplitB[q]][j], d);
                    }
        }
    };
    // (KG = 2: the second group's range is never the longer one; every barrier is for both.)
    const int nk = max(kend - kbeg, 0) / BK;
    const int nk_all = KG == 1 ? nk : (min(kend_wg, kbeg_wg + k_half) - kbeg_wg) / BK;
    const bool rest = kbeg + nk * BK < kend;
    if constexpr (KG == 1) {
        if (nk > 0) {
            load(kbeg, true);
            store(0);
            if (nk > 1) load(kbeg + BK, true);
        }
        barrier();
        for (int kb = 0; kb + 1 < nk; ++kb) {
            multiply(kb & 1, [&]() {
                store((kb + 1) & 1);
                load(kbeg + min(kb + 2, nk - 1) * BK, true);
            });
            barrier();
        }
        if (rest) load(kbeg + nk * BK, false);
        if (nk > 0) multiply((nk - 1) & 1, []() {});
        if (rest) {
            store(nk & 1);
            barrier();
            multiply(nk & 1, []() {});
        }
        barrier();
    } else {
        if (nk_all > 0) {
            if (nk > 0) {
                load(kbeg, true);
                store(0);
                load(kbeg + (nk > 1 ? BK : 0), true);
            }
            barrier();
            for (int kb = 0; kb < nk_all; ++kb) {
                if (kb < nk)
                    multiply(kb & 1, [&]() {
                        store((kb + 1) & 1);
                        load(kbeg + min(kb + 2, nk - 1) * BK, true);
                    });
                barrier();
            }
        }
        if (rest) {
            load(kbeg + nk * BK, false);
            store(0);
        }
        barrier();
        if (rest) multiply(0, []() {});
        barrier();
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NBK; ++j) acc[i][j] = (acc[i][j] + low[i][j]) * kSplitUnscale;
    if constexpr (KG == 2) {  // the second group's sums to the first
        float* sums = reinterpret_cast<float*>(all_lds);  // [register][thread]; free since the last barrier
        if (grp_k == 1) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NBK; ++j)
#pragma unroll
                    for (int r = 0; r < AR; ++r) sums[((i * NBK + j) * AR + r) * NT + tid] = acc[i][j][r];
        }
        __syncthreads();
        if (grp_k == 0) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NBK; ++j)
#pragma unroll
                    for (int r = 0; r < AR; ++r) acc[i][j][r] += sums[((i * NBK + j) * AR + r) * NT + tid];
        }
        __syncthreads();
    }
    // What leaves the range is multiplied again in fp32: infinities and elements that scaled or rounded
    // to bf16 become one, which leave a NaN in the sums, and sums past the scaled range.
    {
        float bad = 0.0f;  // zero as long as every sum is finite (an or of comparisons: 9.8 -> 10.3 us at 9000 x 384 x 64)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NBK; ++j)
#pragma unroll
                for (int r = 0; r < AR; ++r) bad = fmaf(acc[i][j][r], 0.0f, bad);
        if (__syncthreads_or(bad != 0.0f)) {
            clear();
            for (int k = kbeg_wg; k < kend_wg; k += 64 / MT) {
                const int kk = min(k + h, kend_wg - 1);
                const bool in = k + h < kend_wg;
                float av[MB], bv[NBK];
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    const size_t r = min(row0 + wm * WM + MT * i + c, M - 1);
                    av[i] = in ? A[AKC ? r * lda + kk : (size_t)kk * lda + r] : 0.0f;
                }
#pragma unroll
                for (int j = 0; j < NBK; ++j) {
                    const size_t r = min(col0 + wn * WN + MT * j + c, N - 1);
                    bv[j] = in ? B[BKC ? r * ldb + kk : (size_t)kk * ldb + r] : 0.0f;
                }
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NBK; ++j)
                        acc[i][j] = Mfma<MT>::fp32(av[i], bv[j], acc[i][j]);
            }
        }
    }

    // kEpiKV: cache offset of each row of the tile, (sequence * H * T + position) * head_dim.
    __shared__ size_t kv_row[EPI == kEpiKV ? BM : 1];
    if constexpr (EPI == kEpiKV) {
        for (int rr = threadIdx.x; rr < BM; rr += KG * NT) {
            const int gr = min(row0 + rr, M - 1);
            const int sb = gr / kv.rows_per_seq, p = gr - sb * kv.rows_per_seq;
            kv_row[rr] = ((size_t)sb * kv.H * kv.T + p) * kv.hd;
        }
        __syncthreads();
    }
    if (KG == 2 && grp_k == 1) return;
#pragma unroll
    for (int j = 0; j < NBK; ++j) {
        const int gc = col0 + wn * WN + MT * j + c;
        if (gc >= N) continue;
        float* cache = nullptr;  // kEpiKV: this column's place in the K / V caches, row 0
        if constexpr (EPI == kEpiKV) {
            if (gc >= kv.C) {
                const bool is_v = gc >= 2 * kv.C;
                const int cc = gc - (is_v ? 2 * kv.C : kv.C), hh = cc / kv.hd, d = cc - hh * kv.hd;
                cache = (is_v ? kv.vc : kv.kc) + (size_t)hh * kv.T * kv.hd + d;
            }
        }
        // The residual of all the lane's rows first: C may be R, so the compiler cannot move a
        // load above an earlier store itself (one round trip per row otherwise).
        float res[EPI == kEpiResid ? MB : 1][EPI == kEpiResid ? AR : 1];
        if constexpr (EPI == kEpiResid) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < AR; ++r) {
                    const int gr = min(row0 + wm * WM + MT * i + 8 * (r / 4) + 4 * h + (r % 4), M - 1);
                    res[i][r] = R[(size_t)gr * ldr + gc];
                }
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int r = 0; r < AR; ++r) {
                const int lr = wm * WM + MT * i + 8 * (r / 4) + 4 * h + (r % 4), gr = row0 + lr;
                if (gr >= M) continue;
                const float v = acc[i][j][r];
                if constexpr (SPLIT) {
                    partial[((size_t)z * M + gr) * N + gc] = v;
                } else if constexpr (EPI == kEpiKV) {
                    if (cache) cache[kv_row[lr]] = v;
                    else C[(size_t)gr * ldc + gc] = v;
                } else if constexpr (EPI == kEpiGelu) {
                    C[(size_t)gr * ldc + gc] = gelu_ref(v);
                } else if constexpr (EPI == kEpiResid) {
                    C[(size_t)gr * ldc + gc] = res[i][r] + v;
                } else {
                    C[(size_t)gr * ldc + gc] = v;
                }
            }
        }
    }
}

template <int BM, int BN, int BK, int KG, bool AKC, bool BKC, int EPI, bool SPLIT>
int launch(const SplitGemm& g) {
    const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
    constexpr size_t lds = (size_t)KG * 2 * 3 * (BM + BN) * BK * sizeof(uint16_t);  // 48 KB per group
    auto kern = gemm_split_kernel<BM, BN, BK, 2, 2, KG, AKC, BKC, EPI, SPLIT, BM == 128 ? 32 : 16>;
    if constexpr (lds > 64 * 1024)  // each time: the library may have been started on another device since
        FMLH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)tm * tn, 1, SPLIT ? g.splits : g.planes), dim3(256 * KG), lds, g.s, g.A, g.lda,
                       g.a_plane, g.B, g.ldb, g.b_plane, g.C, g.ldc, g.c_plane, g.M, g.N, g.K, g.R, g.ldr, g.kv,
                       g.partial, g.k_per_split, tm, tn);
    FMLH_LAUNCHED("gemm_split_kernel");
    return FMLH_OK;
}

template <int BM, int BN, int BK, int KG, bool AKC, bool BKC>
int by_epilogue(const SplitGemm& g) {
    if constexpr (AKC) {
        if (g.splits > 1) return launch<BM, BN, BK, KG, AKC, BKC, kEpiNone, true>(g);
        switch (g.epi) {
            case kEpiGelu: return launch<BM, BN, BK, KG, AKC, BKC, kEpiGelu, false>(g);
            case kEpiResid: return launch<BM, BN, BK, KG, AKC, BKC, kEpiResid, false>(g);
            case kEpiKV:
                if constexpr (BKC) return launch<BM, BN, BK, KG, AKC, BKC, kEpiKV, false>(g);
                break;
            default: break;
        }
    }
    FMLH_REQUIRE(g.epi == kEpiNone && g.splits == 1, "gemm_split: epilogue %d, %d splits of this layout", g.epi, g.splits);
    return launch<BM, BN, BK, KG, AKC, BKC, kEpiNone, false>(g);
}

template <int BM, int BN, int BK, int KG>
int by_layout(const SplitGemm& g) {
    if (g.a_kc) return g.b_kc ? by_epilogue<BM, BN, BK, KG, true, true>(g) : by_epilogue<BM, BN, BK, KG, true, false>(g);
    return g.b_kc ? by_epilogue<BM, BN, BK, KG, false, true>(g) : by_epilogue<BM, BN, BK, KG, false, false>(g);
}

}  // namespace

bool gemm_split_takes(const SplitGemm& g) {
    // K-contiguous operands are read 16 bytes at a time; a tile's rows (or a K block's) must lie
    // within 32-bit byte offsets of its first element.
    auto vec = [](const float* p, int ld, size_t plane) { return (uintptr_t)p % 16 == 0 && ld % 4 == 0 && plane % 4 == 0; };
    if (g.a_kc && !vec(g.A, g.lda, g.a_plane)) return false;
    if (g.b_kc && !vec(g.B, g.ldb, g.b_plane)) return false;
    return g.M > 0 && g.N > 0 && g.K > 0 && g.lda < (1 << 22) && g.ldb < (1 << 22) && g.planes <= 65535;
}

int gemm_split(const SplitGemm& g) {
    FMLH_REQUIRE(gemm_split_takes(g), "gemm_split: %dx%dx%d, row strides %d and %d: not aligned or too long", g.M, g.N, g.K,
                 g.lda, g.ldb);
    FMLH_REQUIRE(g.splits == 1 || (g.partial && g.k_per_split % 16 == 0), "gemm_split: split K without room");
    if (g.tile == 128) return by_layout<128, 128, 16, 1>(g);
    return g.k_groups == 2 ? by_layout<64, 64, 32, 2>(g) : by_layout<64, 64, 32, 1>(g);
}

}  // namespace fmlh

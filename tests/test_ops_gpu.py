"""GPU parity of the matrix-op entry points (the MatrixHIP<float> overload set).

Each op runs through the C ABI on device memory and is compared with the oracle's
restatement of the reference routine (same fp32 formula) or float64.  Tolerances (normwise,
written per test) cover fp32 reassociation and libm-vs-device exp/erf ulps; data movement ops
(copy, gather, split, fill, argmax) must be exact.
"""
import numpy as np
import pytest

import freeml_amd as fh
import oracle
from plans import SPLIT, plan, strided_tile

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    fh.init(0)
    arch, cus = fh.device_info()
    print(f"device {arch} with {cus} CUs", flush=True)
    assert arch.startswith("gfx950")


D = fh.DeviceArray.from_host


def _rng(s):
    return np.random.default_rng(s)


def _close(got, ref64, tol, scale=None):
    scale = np.max(np.abs(ref64)) if scale is None else scale
    err = np.max(np.abs(got.astype(np.float64) - ref64)) / max(scale, 1e-30)
    assert err <= tol, f"normwise error {err:.3e} > {tol:.1e}"


# Shapes hit: skinny NN/NT (M <= 8), MFMA 64x64 / 128x128 tiles, split-K, ragged edges,
# K not a multiple of 16 (strided fallback).
MUL_SHAPES = [(1, 1152, 384), (4, 1536, 384), (8, 65, 64), (64, 1152, 384), (64, 384, 1536),
              (257, 130, 64), (1024, 512, 768), (37, 50, 65), (3, 7, 5)]


@pytest.mark.parametrize("mode", [fh.NONE, fh.RIGHT, fh.LEFT, fh.BOTH])
@pytest.mark.parametrize("shape", MUL_SHAPES)
def test_mul(mode, shape):
    M, N, K = shape
    print(f"mul mode={mode} M={M} N={N} K={K}", flush=True)
    r = _rng(M * 7 + N + K)
    A = r.standard_normal((M, K)).astype(np.float32)
    B = r.standard_normal((K, N)).astype(np.float32)
    L = np.ascontiguousarray(A.T) if mode in (fh.LEFT, fh.BOTH) else A
    R = np.ascontiguousarray(B.T) if mode in (fh.RIGHT, fh.BOTH) else B
    dL, dR, dO = D(L), D(R), fh.DeviceArray((M, N))
    fh.mul(mode, dO.ptr, dL.ptr, dR.ptr, M, N, K)
    got = dO.numpy()
    ref64 = A.astype(np.float64) @ B.astype(np.float64)
    # fp32 accumulation error bound ~ K * eps * sum|a||b|; normwise against |A||B|.
    absprod = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    _close(got, ref64, 2e-6 * np.sqrt(K) + 1e-6, scale=np.max(absprod))


@pytest.mark.parametrize("epi", [fh.EPI_NONE, fh.EPI_GELU, fh.EPI_RESID])
@pytest.mark.parametrize("shape,bt", [((1, 1536, 384), 0), ((1, 384, 384), 1), ((8, 50304, 768), 1),
                                      ((64, 1152, 384), 0), ((4096, 384, 1536), 0),
                                      ((512, 768, 768), 1), ((64, 65, 384), 1),
                                      # skinny NT on matrix cores: ragged N, the longest K held in
                                      # LDS, and one K past it (per-column kernel)
                                      ((5, 100, 4096), 1), ((8, 768, 3072), 1), ((2, 2304, 768), 1),
                                      ((7, 33, 16), 1), ((3, 40, 4112), 1)])
def test_gemm_ex_epilogues(epi, shape, bt):
    M, N, K = shape
    print(f"gemm_ex epi={epi} M={M} N={N} K={K} bt={bt}", flush=True)
    r = _rng(M + N + K + epi)
    A = (r.standard_normal((M, K)) * 0.5).astype(np.float32)
    W = (r.standard_normal((K, N)) * 0.02).astype(np.float32)
    Rm = r.standard_normal((M, N)).astype(np.float32)
    Wd = np.ascontiguousarray(W.T) if bt else W
    dA, dW, dC, dR = D(A), D(Wd), fh.DeviceArray((M, N)), D(Rm)
    fh.gemm_ex(dA.ptr, K, dW.ptr, K if bt else N, bt, dC.ptr, N, M, N, K, epi,
               dR.ptr if epi == fh.EPI_RESID else 0, N)
    got = dC.numpy()
    acc = A.astype(np.float64) @ W.astype(np.float64)
    if epi == fh.EPI_GELU:
        from scipy.special import erf
        ref = 0.5 * acc * (1 + erf(acc / np.sqrt(2)))
    elif epi == fh.EPI_RESID:
        ref = Rm + acc
    else:
        ref = acc
    _close(got, ref, 1e-5)


_NT_REF = {}


def _nt_case(M, N, K, seed):
    key = (M, N, K, seed)
    if key not in _NT_REF:
        r = _rng(seed)
        A = (r.standard_normal((M, K)) * 0.5).astype(np.float32)
        Wt = (r.standard_normal((N, K)) * 0.05).astype(np.float32)
        Rm = r.standard_normal((M, N)).astype(np.float32)
        _NT_REF[key] = (A, Wt, Rm, A.astype(np.float64) @ Wt.T.astype(np.float64))
    return _NT_REF[key]


# B stored N x K on the split tiles: ragged M and N (clamped edge rows), K of 1, 2, 3 and many 16-wide
# blocks (the pipeline's start and end), either tile (forced through FMLH_GEMM_NT_TILE) and the choice.
@pytest.mark.parametrize("tile", ["", "128x128", "64x64"])
@pytest.mark.parametrize("shape", [(1000, 1030, 384), (300, 2000, 48), (520, 2100, 16),
                                   (1100, 700, 32), (4096, 2304, 768)])
def test_gemm_nt_kernel_tiles(tile, shape, monkeypatch):
    M, N, K = shape
    print(f"gemm nt tile={tile or 'default'} M={M} N={N} K={K}", flush=True)
    if tile:
        monkeypatch.setenv("FMLH_GEMM_NT_TILE", tile)
    p = plan(M, N, K, 1)
    assert p.kind == SPLIT and (not tile or p.tile == int(tile[:tile.index("x")])), p
    A, Wt, Rm, acc = _nt_case(M, N, K, 11)
    dA, dW, dC = D(A), D(Wt), fh.DeviceArray((M, N))
    fh.gemm_ex(dA.ptr, K, dW.ptr, K, 1, dC.ptr, N, M, N, K, fh.EPI_NONE, 0, N)
    _close(dC.numpy(), acc, 1e-5)


# Launches of the split tiles: 64 x 64 with one and with two groups of waves, K ranges, 128 x 128.
SPLIT_LAUNCHES = [((1100, 900, 64), "", (64, 1, 1)), ((700, 600, 400), "", (64, 2, 1)), ((300, 260, 1600), "", (64, 2, 10)),
                  ((700, 600, 400), "128x128", (128, 1, 1))]


def _split_launch(shape, tile, launch, bt, monkeypatch):
    """Checks that a product takes the split tiles as meant, whatever the planner has become."""
    if tile:
        monkeypatch.setenv("FMLH_GEMM_NT_TILE", tile)
    p = plan(*shape, bt)
    assert p.kind == SPLIT and launch in (None, (p.tile, p.k_groups, p.splits)), p


def _gemm_ex(A, W, bt):
    (M, K), N = A.shape, W.shape[1]
    dA, dW, dC = D(A), D(np.ascontiguousarray(W.T) if bt else W), fh.DeviceArray((M, N))
    fh.gemm_ex(dA.ptr, K, dW.ptr, K if bt else N, bt, dC.ptr, N, M, N, K, fh.EPI_NONE, 0, N)
    return dC.numpy().astype(np.float64)


def _split_error_ok(got, A64, W64):
    """Element by element: every 8 k of the six part products round once (6 K / 8 roundings of 2^-24 on sums
    below |A||B|), the parts left out are below 2^-24.  As a whole: the roundings grow as the root of K
    (1.1e-7, 1.6e-7 and 3.4e-7 measured at K 384, 768 and 3072, 1.3e-6 at 20016), while without any one of
    the small part products the error is 2.4e-6 and more at every K: twice the first, at most two
    thirds of the second."""
    K, ref = A64.shape[1], A64 @ W64
    err = got - ref
    assert np.all(np.abs(err) <= (0.75 * K + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(W64)))
    assert np.linalg.norm(err) <= min(1.5e-8 * np.sqrt(K) + 6e-8, 1.6e-6) * np.linalg.norm(ref)


# Products on the bf16 matrix cores (operands split into three bf16 parts): one row and column past a
# tile, one K block and the remainder of the wide tile's, both tiles and both layouts of B.
@pytest.mark.parametrize("tile", ["128x128", "64x64"])
@pytest.mark.parametrize("bt", [0, 1])
# (from the fifth on, on 64 x 64 tiles: two groups of waves, with equal, unequal and ragged parts of K; the
# last three in K ranges too)
@pytest.mark.parametrize("shape", [(65, 8300, 16), (4097, 129, 48), (1100, 901, 64), (130, 4300, 80), (321, 449, 128),
                                   (449, 385, 144), (450, 386, 160), (385, 513, 400), (200, 96, 1008), (520, 390, 1008),
                                   (66, 66, 4112)])
def test_gemm_split_bf16_edges(shape, bt, tile, monkeypatch):
    M, N, K = shape
    print(f"split gemm tile={tile} M={M} N={N} K={K} bt={bt}", flush=True)
    _split_launch(shape, tile, None, bt, monkeypatch)
    p = plan(*shape, bt)
    assert p.tile == int(tile[:tile.index("x")]) and (tile == "128x128" or p.k_groups == 1 + (K >= 128))
    assert (p.splits > 1) == (K > 1000)
    r = _rng(M + N + K)
    A = r.standard_normal((M, K)).astype(np.float32)
    W = (r.standard_normal((K, N)) * np.exp2(r.integers(-12, 12, (K, N)))).astype(np.float32)
    _split_error_ok(_gemm_ex(A, W, bt), A.astype(np.float64), W.astype(np.float64))


# Operands the bf16 parts cannot carry take the fp32 path inside the kernel: infinities, NaN and
# elements near fp32's end give what fp32 arithmetic gives; rows of tiny elements keep their accuracy.
@pytest.mark.parametrize("bt", [0, 1])
@pytest.mark.parametrize("shape,tile,launch", SPLIT_LAUNCHES)
def test_gemm_split_bf16_special_values(shape, tile, launch, bt, monkeypatch):
    print(f"special values {shape} {tile} bt={bt}", flush=True)
    _split_launch(shape, tile, launch, bt, monkeypatch)
    M, N, K = shape
    r = _rng(5)
    A = r.standard_normal((M, K)).astype(np.float32)
    W = r.standard_normal((K, N)).astype(np.float32)
    A[3, 7] = np.inf
    A[150, 0], A[151, 5] = -np.inf, np.nan
    A[290, 9] = 3.4e38  # rounds to an infinity in bf16
    A[200, K - 1] = 1e33  # past the scaled range
    W[:, 130] *= np.float32(1e-34)
    A[70, :] *= np.float32(1e-33)
    W[7, 11] = 0.0  # infinity times zero
    got = _gemm_ex(A, W, bt)
    with np.errstate(all="ignore"):
        ref = A.astype(np.float64) @ W.astype(np.float64)
        ref[np.abs(ref) > np.finfo(np.float32).max] = np.inf * np.sign(ref[np.abs(ref) > np.finfo(np.float32).max])
        prod = np.abs(A.astype(np.float64)) @ np.abs(W.astype(np.float64))
    # the row whose partial sums lie at the end of fp32's range may overflow either way
    ok = np.ones((M, N), bool)
    ok[290] = np.abs(prod[290]) < 1e38
    fin = np.isfinite(ref) & ok
    assert np.array_equal(np.isnan(got)[ok], np.isnan(ref)[ok])
    assert np.array_equal(got[ok & np.isinf(ref)], ref[ok & np.isinf(ref)])
    # (2^-149: sums that are subnormal themselves, 1e-34 times 1e-33)
    assert np.all(np.abs(got[fin] - ref[fin]) <= (0.75 * K + 8) * (2.0 ** -24 * prod[fin] + 2.0 ** -149))


# Sums within 2^-8 of fp32's largest number: a0 b0 alone is past it where both bf16 parts are rounded
# up.  One such element per row of A, its partner in B, everything else small.
@pytest.mark.parametrize("bt", [0, 1])
@pytest.mark.parametrize("shape,tile,launch", SPLIT_LAUNCHES)
def test_gemm_split_near_the_largest_number(shape, tile, launch, bt, monkeypatch):
    print(f"near the largest number {shape} {tile} bt={bt}", flush=True)
    _split_launch(shape, tile, launch, bt, monkeypatch)
    M, N, K = shape
    r = _rng(K)
    A, W = (r.standard_normal((M, K)) * 1e-3).astype(np.float32), (r.standard_normal((K, N)) * 1e-3).astype(np.float32)
    A[:, 5], W[5, :] = 0.0, 0.0
    A[::3, 5] = W[5, ::2] = np.float32(1.998 * 2.0 ** 63)  # bf16: 2^64
    A64, W64 = A.astype(np.float64), W.astype(np.float64)
    ref = A64 @ W64
    assert 0.99 * 2.0 ** 128 < np.abs(ref).max() < np.finfo(np.float32).max
    assert np.all(np.abs(_gemm_ex(A, W, bt) - ref) <= (0.75 * K + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(W64)))


# A tiny element (of A, of B, of both; down to fp32's subnormals) in rows of normal ones, where it
# meets a large partner and the other elements meet zeros: as accurate as anywhere else.  Every other
# column has normal partners beside the tiny ones.
@pytest.mark.parametrize("bt", [0, 1])
@pytest.mark.parametrize("shape,tile,launch", SPLIT_LAUNCHES)
def test_gemm_split_tiny_elements_beside_normal_ones(shape, tile, launch, bt, monkeypatch):
    _split_launch(shape, tile, launch, bt, monkeypatch)
    M, N, K = shape
    for t in (-98, -103, -110, -118, -126, -140):
        print(f"tiny elements 2^{t} {shape} {tile} bt={bt}", flush=True)
        r = _rng(K - t)
        A, W = r.standard_normal((M, K)), r.standard_normal((K, N))
        A[::2, 7] *= 2.0 ** t
        W[:, ::2] = 0
        W[7, ::2] = r.standard_normal((N + 1) // 2) * 2.0 ** 60
        A[5::32, :] = 0
        A[5::32, 9] = r.standard_normal(len(range(5, M, 32))) * 2.0 ** 40
        W[9, 1::32] *= 2.0 ** t
        A, W = A.astype(np.float32), W.astype(np.float32)
        A64, W64 = A.astype(np.float64), W.astype(np.float64)
        err, prod = np.abs(_gemm_ex(A, W, bt) - A64 @ W64), np.abs(A64) @ np.abs(W64)
        # (2^-149: sums that are subnormal themselves)
        assert np.all(err <= (0.75 * K + 8) * (2.0 ** -24 * prod + 2.0 ** -149)), t


def test_matmul_strided_split_tiny_elements_beside_normal_ones():
    M, N, K = 600, 500, 130
    assert strided_tile(fh.LEFT, M, N, K, M, 1, N, 1, N, 1) == 64
    r = _rng(2)
    A, W = r.standard_normal((M, K)), r.standard_normal((K, N))
    A[:, 7] *= 2.0 ** -120
    W[:, ::2] = 0
    W[7, ::2] = 2.0 ** 60
    A, W = A.astype(np.float32), W.astype(np.float32)
    dA, dW, dC = D(np.ascontiguousarray(A.T)), D(W), fh.DeviceArray((M, N))
    fh.matmul_strided(fh.LEFT, dC.ptr, dA.ptr, dW.ptr, M, N, K, M, 1, N, 1, N, 1)
    A64, W64 = A.astype(np.float64), W.astype(np.float64)
    assert np.all(np.abs(dC.numpy() - A64 @ W64) <= (0.75 * K + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(W64)))


# Many K ranges (the last one short or ragged) and partials beyond the no-alloc array (1000 x 770 in 6
# or more ranges).  (The rounding per range is within the bounds' slack for eight k.)
@pytest.mark.parametrize("mode", [fh.NONE, fh.RIGHT])
@pytest.mark.parametrize("shape", [(65, 129, 8208), (130, 96, 5008), (1000, 770, 5008), (257, 770, 20016)])
def test_mul_many_k_ranges(shape, mode):
    M, N, K = shape
    print(f"mul mode={mode} {shape}", flush=True)
    r = _rng(M + N)
    A, W = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    dA, dW, dC = D(A), D(np.ascontiguousarray(W.T) if mode == fh.RIGHT else W), fh.DeviceArray((M, N))
    fh.mul(mode, dC.ptr, dA.ptr, dW.ptr, M, N, K)
    p = plan(M, N, K, int(mode == fh.RIGHT))
    assert p.kind == SPLIT and p.splits >= 3, p
    _split_error_ok(dC.numpy(), A.astype(np.float64), W.astype(np.float64))


@pytest.mark.parametrize("mode", [fh.NONE, fh.RIGHT])
@pytest.mark.parametrize("shape,splits", [((70, 64, 33008), 47), ((130, 192, 16400), 24), ((66, 64, 131072), 64)])
def test_mul_more_than_16_k_ranges(shape, splits, mode):
    """Bound: as above, with a rounding per range; and 2-norm errors of fp32 sums of K / splits terms."""
    M, N, K = shape
    p = plan(M, N, K, int(mode == fh.RIGHT))
    print(f"mul mode={mode} {shape} {p}", flush=True)
    assert p.kind == SPLIT and p.splits == splits
    r = _rng(M + N)
    A, W = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((K, N), dtype=np.float32)
    dA, dW, dC = D(A), D(np.ascontiguousarray(W.T) if mode == fh.RIGHT else W), fh.DeviceArray((M, N))
    fh.mul(mode, dC.ptr, dA.ptr, dW.ptr, M, N, K)
    A64, W64 = A.astype(np.float64), W.astype(np.float64)
    err, ref = dC.numpy() - A64 @ W64, A64 @ W64
    assert np.all(np.abs(err) <= (0.75 * K + 8 + splits) * 2.0 ** -24 * (np.abs(A64) @ np.abs(W64)))
    assert np.linalg.norm(err) <= 4e-7 * np.linalg.norm(ref)


# Row strides of 2^22 floats and more: past the split tiles' 32-bit offsets, on the fp32 tiles.
@pytest.mark.parametrize("M,N,K,bt,lda,ldb", [(1000, 1000, 32, 0, 32, 1 << 22), (130, 4096, 32, 0, 1 << 22, 4096),
                                              (130, 4096, 32, 1, (1 << 22) + 4, 32), (4096, 130, 32, 1, 32, 1 << 22)])
@pytest.mark.parametrize("epi", [fh.EPI_NONE, fh.EPI_RESID])
def test_gemm_ex_long_row_strides(M, N, K, bt, lda, ldb, epi):
    print(f"gemm_ex M={M} N={N} K={K} bt={bt} lda={lda} ldb={ldb} epi={epi}", flush=True)
    r = _rng(M + N)
    A, W = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    Rm = r.standard_normal((M, N)).astype(np.float32)

    def rows(X, ld):
        d = fh.DeviceArray(X.shape[0] * ld)
        for i, row in enumerate(np.ascontiguousarray(X)):
            fh.call("fmlh_memcpy_h2d", d.at(i * ld), row.ctypes.data, row.nbytes)
        return d

    dA, dW, dC = rows(A, lda), rows(W.T if bt else W, ldb), D(Rm)
    fh.gemm_ex(dA.ptr, lda, dW.ptr, ldb, bt, dC.ptr, N, M, N, K, epi, dC.ptr if epi == fh.EPI_RESID else 0, N)
    _close(dC.numpy(), A.astype(np.float64) @ W + (Rm if epi == fh.EPI_RESID else 0), 1e-5)


def test_mul_4m_columns():
    M, N, K = 65, 1 << 22, 16
    r = _rng(9)
    A, W = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N), dtype=np.float32)
    dA, dW, dC = D(A), D(W), fh.DeviceArray((M, N))
    fh.mul(fh.NONE, dC.ptr, dA.ptr, dW.ptr, M, N, K)
    got, cols = dC.numpy(), np.r_[0:200, r.integers(0, N, 2000), N - 200:N]
    _close(got[:, cols], A.astype(np.float64) @ W[:, cols], 1e-5)


# Strided products of 64 tiles' worth of outputs and more (the split bf16 tiles): every mode, both
# index orders of each operand (rows or columns contiguous), batched planes, K with a remainder,
# row strides that keep 16-byte rows and ones that do not (the wave-split kernel), 128-wide tiles.
@pytest.mark.parametrize("mode", [fh.NONE, fh.RIGHT, fh.LEFT, fh.BOTH])
@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("shape", [(190, 333, 37, 5, 3), (190, 333, 37, 5, 2), (129, 65, 100, 33, 0), (300, 260, 20, 86, 4),
                                   (520, 510, 131, 1, 0), (65, 2100, 205, 2, 1)])
def test_matmul_strided_split_tiles(shape, swap, mode):
    M, N, K, planes, pad = shape
    print(f"strided split mode={mode} swap={swap} {shape}", flush=True)
    r = _rng(M + K + mode)
    A = r.standard_normal((planes, M, K)).astype(np.float32)
    B = r.standard_normal((planes, K, N)).astype(np.float32)

    def stored(X, transposed):  # as (stored array, plane, row stride, column stride) of X's mode view
        V = np.swapaxes(X, 1, 2) if transposed else X  # the matrix the call names
        S = np.swapaxes(V, 1, 2) if swap else V         # how it lies in memory
        ld = S.shape[2] + (-S.shape[2]) % 4 + pad
        P = np.zeros((planes, S.shape[1], ld), np.float32)
        P[:, :, :S.shape[2]] = S
        return P, P.shape[1] * ld, *((1, ld) if swap else (ld, 1))

    L, lp, lrs, lcs = stored(A, mode in (fh.LEFT, fh.BOTH))
    R, rp, rrs, rcs = stored(B, mode in (fh.RIGHT, fh.BOTH))
    a_kc, b_kc = (mode in (fh.LEFT, fh.BOTH)) == swap, (mode in (fh.RIGHT, fh.BOTH)) != swap
    tile = strided_tile(mode, M, N, K, lrs, lcs, rrs, rcs, N + 3, 1, planes, lp, rp)
    assert (tile > 0) == (pad % 4 == 0 or not (a_kc or b_kc)), tile
    dL, dR, dO = D(L), D(R), D(np.full((planes, M, N + 3), 7.0, np.float32))
    fh.matmul_strided(mode, dO.ptr, dL.ptr, dR.ptr, M, N, K, lrs, lcs, rrs, rcs, N + 3, 1, planes, lp, rp, M * (N + 3))
    got = dO.numpy()
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(got[:, :, :N] - A64 @ B64) <= (0.75 * K + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)))
    assert np.all(got[:, :, N:] == 7.0)


# Many small planes: 64 x 64 tiles, however many there are, but the vector kernel for quarters of one.
@pytest.mark.parametrize("mode", [fh.NONE, fh.RIGHT, fh.LEFT])
@pytest.mark.parametrize("M,N,K", [(16, 64, 256), (64, 28, 16), (24, 72, 64), (48, 64, 64), (32, 28, 64)])
def test_matmul_strided_many_small_planes(M, N, K, mode):
    planes = 600
    r = _rng(M + K)
    A = r.standard_normal((planes, M, K), dtype=np.float32)
    B = r.standard_normal((planes, K, N), dtype=np.float32)
    L = np.ascontiguousarray(np.swapaxes(A, 1, 2) if mode == fh.LEFT else A)
    R = np.ascontiguousarray(np.swapaxes(B, 1, 2) if mode == fh.RIGHT else B)
    dL, dR, dO = D(L), D(R), fh.DeviceArray((planes, M, N))
    args = (mode, M, N, K, L.shape[2], 1, R.shape[2], 1, N, 1, planes, M * K, K * N)
    assert strided_tile(*args) == (0 if M == 32 else 64)
    fh.matmul_strided(mode, dO.ptr, dL.ptr, dR.ptr, *args[1:], M * N)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(dO.numpy() - A64 @ B64) <= (0.75 * K + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)))


@pytest.mark.parametrize("epi", [fh.EPI_GELU, fh.EPI_RESID])
@pytest.mark.parametrize("tile", ["128x128", "64x64"])
def test_gemm_nt_kernel_epilogues_in_place(epi, tile, monkeypatch):
    M, N, K = 1000, 1030, 384
    print(f"gemm nt epi={epi} tile={tile}", flush=True)
    monkeypatch.setenv("FMLH_GEMM_NT_TILE", tile)
    A, Wt, Rm, acc = _nt_case(M, N, K, 11)
    dA, dW, dX = D(A), D(Wt), D(Rm)
    if epi == fh.EPI_RESID:  # C aliases R, as the block's residual add does
        fh.gemm_ex(dA.ptr, K, dW.ptr, K, 1, dX.ptr, N, M, N, K, epi, dX.ptr, N)
        ref = Rm + acc
    else:
        fh.gemm_ex(dA.ptr, K, dW.ptr, K, 1, dX.ptr, N, M, N, K, epi, 0, N)
        from scipy.special import erf
        ref = 0.5 * acc * (1 + erf(acc / np.sqrt(2)))
    _close(dX.numpy(), ref, 1e-5)


@pytest.mark.parametrize("epi", [fh.EPI_NONE, fh.EPI_GELU, fh.EPI_RESID])
@pytest.mark.parametrize("bt", [0, 1])
@pytest.mark.parametrize("shape", [(4096, 384, 1536), (2000, 332, 1056)])
def test_gemm_split_k_ranges_with_epilogues(shape, bt, epi, monkeypatch):
    """Split products in one, two and five K ranges (FMLH_GEMM_NT_SPLIT_K; the last of five is short):
    partials and the reduction with the epilogue, the residual in place, agree to fp32 rounding."""
    M, N, K = shape
    print(f"gemm K ranges epi={epi} M={M} N={N} K={K} bt={bt}", flush=True)
    A, Wt, Rm, acc = _nt_case(M, N, K, 5)
    dA, dW = D(A), D(Wt if bt else np.ascontiguousarray(Wt.T))
    outs = []
    for ranges in ("0", "2", "5"):
        monkeypatch.setenv("FMLH_GEMM_NT_SPLIT_K", ranges)
        p = plan(M, N, K, bt)
        assert p.kind == SPLIT and p.splits == max(1, int(ranges)), p
        dX = D(Rm)
        fh.gemm_ex(dA.ptr, K, dW.ptr, K if bt else N, bt, dX.ptr, N, M, N, K, epi, dX.ptr if epi == fh.EPI_RESID else 0, N)
        outs.append(dX.numpy())
    if epi == fh.EPI_RESID:
        ref = Rm + acc
    elif epi == fh.EPI_GELU:
        from scipy.special import erf
        ref = 0.5 * acc * (1 + erf(acc / np.sqrt(2)))
    else:
        ref = acc
    for got in outs:
        _close(got, ref, 1e-6)  # K 1536: 2.4e-7 of the sums' 2-norm, a largest of four times that


@pytest.mark.parametrize("bt", [0, 1])
def test_split_k_products_back_to_back(bt):
    """Split-K products (batched-decode shapes) reduce in the launch: the last split of each
    tile adds the partials and resets the tile's arrival counter.  Several products in a row,
    of different tile counts and split factors, each with fresh inputs, must all be right (a
    counter left non-zero would skip a tile's reduction in the next product)."""
    r = _rng(17 + bt)
    shapes = [(64, 1152, 384, fh.EPI_NONE), (64, 384, 1536, fh.EPI_RESID), (64, 1152, 384, fh.EPI_NONE),
              (48, 1536, 384, fh.EPI_GELU), (64, 384, 1536, fh.EPI_RESID), (64, 1152, 384, fh.EPI_NONE)]
    for rep, (M, N, K, epi) in enumerate(shapes * 4):
        print(f"split-K product {rep}: M={M} N={N} K={K} epi={epi} bt={bt}", flush=True)
        A = (r.standard_normal((M, K)) * 0.5).astype(np.float32)
        W = (r.standard_normal((K, N)) * 0.05).astype(np.float32)
        X = r.standard_normal((M, N)).astype(np.float32)
        dA, dW, dX = D(A), D(np.ascontiguousarray(W.T) if bt else W), D(X)
        fh.gemm_ex(dA.ptr, K, dW.ptr, K if bt else N, bt, dX.ptr, N, M, N, K, epi,
                   dX.ptr if epi == fh.EPI_RESID else 0, N)
        acc = A.astype(np.float64) @ W.astype(np.float64)
        if epi == fh.EPI_RESID:
            ref = X + acc
        elif epi == fh.EPI_GELU:
            from scipy.special import erf
            ref = 0.5 * acc * (1 + erf(acc / np.sqrt(2)))
        else:
            ref = acc
        _close(dX.numpy(), ref, 1e-5)


def test_gemm_ex_residual_in_place():
    M, N, K = 16, 384, 384
    r = _rng(5)
    A = r.standard_normal((M, K)).astype(np.float32)
    W = (r.standard_normal((N, K)) * 0.02).astype(np.float32)
    X = r.standard_normal((M, N)).astype(np.float32)
    dA, dW, dX = D(A), D(W), D(X)
    fh.gemm_ex(dA.ptr, K, dW.ptr, K, 1, dX.ptr, N, M, N, K, fh.EPI_RESID, dX.ptr, N)
    _close(dX.numpy(), X + A.astype(np.float64) @ W.T.astype(np.float64), 1e-5)


@pytest.mark.parametrize("T,C,H", [(64, 64, 4), (256, 384, 6), (200, 96, 3)])
def test_matmul_strided_attention_views(T, C, H):
    """The per-head views of CausalSelfAttentionLayer.h:430-497: Q_h K_h^T with row stride C,
    then P V_h written into a column slice of Y (K = T: past one 64-wide chunk for T > 64),
    and the backward's transposed-left products P^T dY_h and dS^T Q_h (:612-660)."""
    hd = C // H
    r = _rng(9)
    Q = r.standard_normal((T, C)).astype(np.float32)
    K = r.standard_normal((T, C)).astype(np.float32)
    V = r.standard_normal((T, C)).astype(np.float32)
    dQ, dK, dV = D(Q), D(K), D(V)
    dS, dY = fh.DeviceArray((H, T, T)), fh.DeviceArray((T, C))
    for h in range(H):
        fh.matmul_strided(fh.RIGHT, dS.at(h * T * T), dQ.at(h * hd), dK.at(h * hd), T, T, hd,
                          C, 1, C, 1, T, 1)
    S = dS.numpy()
    for h in range(H):
        ref = Q[:, h * hd:(h + 1) * hd].astype(np.float64) @ K[:, h * hd:(h + 1) * hd].T.astype(np.float64)
        _close(S[h], ref, 1e-6)
    P = np.abs(S[0]) / np.abs(S[0]).sum(1, keepdims=True)
    dP = D(P.astype(np.float32))
    for h in range(H):
        fh.matmul_strided(fh.NONE, dY.at(h * hd), dP.ptr, dV.at(h * hd), T, hd, T, T, 1, C, 1, C, 1)
    Y = dY.numpy()
    for h in range(H):
        _close(Y[:, h * hd:(h + 1) * hd], P.astype(np.float64) @ V[:, h * hd:(h + 1) * hd], 1e-6)
    # dV_h = P^T dY_h: Left mode, L = P (T x T, row stride T), R = a column slice of Y.
    dVh = fh.DeviceArray((H, T, hd))
    for h in range(H):
        fh.matmul_strided(fh.LEFT, dVh.at(h * T * hd), dP.ptr, dY.at(h * hd), T, hd, T, T, 1, C, 1, hd, 1)
    G = dVh.numpy()
    for h in range(H):
        _close(G[h], P.astype(np.float64).T @ Y[:, h * hd:(h + 1) * hd].astype(np.float64), 1e-6)


@pytest.mark.parametrize("M,N,K", [(20, 30, 40), (70, 33, 300)])
def test_matmul_strided_batched_planes(M, N, K):
    r = _rng(10)
    B = 3
    A = r.standard_normal((B, M, K)).astype(np.float32)
    Bm = r.standard_normal((B, N, K)).astype(np.float32)
    dA, dB, dO = D(A), D(Bm), fh.DeviceArray((B, M, N))
    fh.matmul_strided(fh.RIGHT, dO.ptr, dA.ptr, dB.ptr, M, N, K, K, 1, K, 1, N, 1, B, M * K, N * K, M * N)
    ref = np.einsum("bmk,bnk->bmn", A.astype(np.float64), Bm.astype(np.float64))
    _close(dO.numpy(), ref, 1e-6)


@pytest.mark.parametrize("mode", [fh.NONE, fh.LEFT, fh.RIGHT, fh.BOTH])
@pytest.mark.parametrize("M,N,K", [(6, 5, 7), (40, 33, 70), (64, 64, 64)])
def test_matmul_strided_against_oracle_all_modes(mode, M, N, K):
    """fmlh_matmul_strided on operands read through element strides (row strides wider than
    the row, column strides > 1, a column-strided output) against the oracle's MulStrided
    restatement (bit-exact to the compiled reference); elements of the output buffer the product
    does not address keep their contents."""
    r = _rng(100 + mode)
    tl, tr = mode in (fh.LEFT, fh.BOTH), mode in (fh.RIGHT, fh.BOTH)
    a_rows, a_cols = (K, M) if tl else (M, K)
    b_rows, b_cols = (N, K) if tr else (K, N)
    a_cs, b_cs, c_cs = 2, 3, 2
    a_rs, b_rs, c_rs = a_cols * a_cs + 5, b_cols * b_cs + 1, N * c_cs + 3
    A = r.standard_normal(a_rows * a_rs).astype(np.float32)
    B = r.standard_normal(b_rows * b_rs).astype(np.float32)
    ref = oracle.mul_strided(mode, A, B, M, N, K, a_rs, a_cs, b_rs, b_cs, c_rs, c_cs, M * c_rs)
    dA, dB = D(A), D(B)
    dO = D(np.zeros(M * c_rs, np.float32))
    fh.matmul_strided(mode, dO.ptr, dA.ptr, dB.ptr, M, N, K, a_rs, a_cs, b_rs, b_cs, c_rs, c_cs)
    got = dO.numpy()
    assert np.max(np.abs(got - ref)) <= 1e-5 * max(1.0, np.max(np.abs(ref)))
    written = np.zeros(M * c_rs, bool)
    for i in range(M):
        written[i * c_rs + np.arange(N) * c_cs] = True
    assert not got[~written].any()


@pytest.mark.parametrize("rows,cols", [(1, 64), (256, 256), (5, 4096), (3, 65)])
def test_softmax(rows, cols):
    r = _rng(rows + cols)
    x = (r.standard_normal((rows, cols)) * 3).astype(np.float32)
    if cols >= 64:
        x = oracle.scale_add(x, 0.125, oracle.triangle_lower(rows, cols, 0.0, -np.inf))
    dX, dO = D(x), fh.DeviceArray((rows, cols))
    fh.softmax(dO.ptr, dX.ptr, rows, cols)
    got = dO.numpy()
    ref = oracle.softmax(x)
    np.testing.assert_allclose(got, ref, rtol=5e-6, atol=1e-9)
    assert np.all(got[np.isinf(x)] == 0.0)


@pytest.mark.parametrize("rows,cols,beta", [(1, 384, False), (300, 768, True), (7, 64, False), (2, 100, True)])
def test_layernorm(rows, cols, beta):
    r = _rng(rows * cols)
    x = (r.standard_normal((rows, cols)) * 2 + 0.3).astype(np.float32)
    g = (1 + 0.1 * r.standard_normal(cols)).astype(np.float32)
    b = r.standard_normal(cols).astype(np.float32) if beta else None
    dX, dG, dO, dH = D(x), D(g), fh.DeviceArray((rows, cols)), fh.DeviceArray((rows, cols))
    dB = D(b) if beta else None
    fh.layernorm(dO.ptr, dX.ptr, dG.ptr, dB.ptr if beta else 0, dH.ptr, rows, cols)
    ref = oracle.layernorm(x, g, b)
    np.testing.assert_allclose(dO.numpy(), ref, rtol=1e-5, atol=2e-6)
    np.testing.assert_allclose(dH.numpy(), oracle.layernorm(x, np.ones(cols, np.float32)), rtol=1e-5, atol=2e-6)


def test_gelu_and_elementwise():
    r = _rng(12)
    n = 100_003
    x = (r.standard_normal(n) * 3).astype(np.float32)
    y = r.standard_normal(n).astype(np.float32)
    dx, dy, do = D(x), D(y), fh.DeviceArray(n)
    fh.gelu(do.ptr, dx.ptr, n)
    np.testing.assert_allclose(do.numpy(), oracle.gelu(x), rtol=2e-6, atol=5e-7)
    fh.add(do.ptr, dx.ptr, dy.ptr, n)
    np.testing.assert_array_equal(do.numpy(), x + y)
    fh.per_element_mul(do.ptr, dx.ptr, dy.ptr, n)
    np.testing.assert_array_equal(do.numpy(), x * y)
    fh.scale_scalar(do.ptr, dx.ptr, 0.25, n)
    np.testing.assert_array_equal(do.numpy(), x * np.float32(0.25))
    s = D(np.array([1.5], np.float32))
    fh.scale(do.ptr, dx.ptr, s.ptr, n)
    np.testing.assert_array_equal(do.numpy(), x * np.float32(1.5))
    fh.fill(do.ptr, 2.5, n)
    np.testing.assert_array_equal(do.numpy(), np.full(n, 2.5, np.float32))
    fh.fill_from(do.ptr, s.ptr, n)
    np.testing.assert_array_equal(do.numpy(), np.full(n, 1.5, np.float32))
    fh.copy(do.ptr, dy.ptr, n)
    np.testing.assert_array_equal(do.numpy(), y)
    m = D(oracle.triangle_lower(1, n, 0.0, -np.inf)[0])
    fh.scale_add(do.ptr, dx.ptr, s.ptr, m.ptr, n)
    np.testing.assert_array_equal(do.numpy(), oracle.scale_add(x, 1.5, oracle.triangle_lower(1, n, 0.0, -np.inf)[0]))
    bias = r.standard_normal(7).astype(np.float32)
    db = D(bias)
    fh.broadcast_add(do.ptr, dx.ptr, db.ptr, 7 * 1000, 7)
    np.testing.assert_array_equal(do.numpy()[:7000], x[:7000] + np.tile(bias, 1000))


def test_gather_split_argmax():
    r = _rng(13)
    V, C, T = 65, 64, 33
    W = r.standard_normal((V, C)).astype(np.float32)
    ids = r.integers(0, V, size=(2, T)).astype(np.float32)
    ids[1, 3] = V + 5  # out of range -> zero row
    dW, dI, dO = D(W), D(ids), fh.DeviceArray((2, T, C))
    fh.gather_rows(dO.ptr, dW.ptr, dI.ptr, C, T, 2, V, 1)
    got = dO.numpy()
    exp = W[np.minimum(ids.astype(np.int64), V - 1)]
    exp[1, 3] = 0.0
    np.testing.assert_array_equal(got, exp)
    # In-range rows against the oracle's GatherRows restatement (bit-exact to the reference).
    np.testing.assert_array_equal(got[0], oracle.gather_rows(W, ids[0]))
    keep = np.arange(T) != 3
    np.testing.assert_array_equal(got[1][keep], oracle.gather_rows(W, ids[1][keep]))
    packed = r.standard_normal((T, 3 * C)).astype(np.float32)
    dp = D(packed)
    q, k, v = (fh.DeviceArray((T, C)) for _ in range(3))
    fh.split_qkv(q.ptr, k.ptr, v.ptr, dp.ptr, T, C)
    np.testing.assert_array_equal(q.numpy(), packed[:, :C])
    np.testing.assert_array_equal(k.numpy(), packed[:, C:2 * C])
    np.testing.assert_array_equal(v.numpy(), packed[:, 2 * C:])
    logits = r.standard_normal((9, 50304)).astype(np.float32)
    logits[2, 10] = logits[2, 40000] = 99.0  # tie: first index wins
    logits[5, :] = 1.0
    dl, di = D(logits), fh.DeviceArray(9, np.int32)
    fh.row_argmax(di.ptr, dl.ptr, 9, 50304)
    got = di.numpy()
    exp = [oracle.argmax(row) for row in logits]
    assert got.tolist() == exp
    assert got[2] == 10 and got[5] == 0


def test_bad_arguments_raise():
    with pytest.raises(fh.FreeMLHipError):
        fh.mul(7, 0, 0, 0, 1, 1, 1)
    a = fh.DeviceArray(4)
    with pytest.raises(fh.FreeMLHipError):
        fh.gemm_ex(a.ptr, 2, a.ptr, 2, 0, a.ptr, 2, 2, 2, 2, fh.EPI_RESID, 0, 2)

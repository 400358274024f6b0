"""Plans of the products, on the host (256 CUs where there is no device)."""
import random

import freeml_amd as fh
from plans import MFMA, SPLIT, engine_workspace, plan, strided_tile


def test_engine_workspace_holds_every_product_of_a_prefill():
    """A prefill runs the blocks on batch x P rows and the lm_head on the batch's last rows; fewer
    rows can plan more K ranges (vocabulary 8192, width 768: 50 rows take 2, 64 take none)."""
    rng = random.Random(3)
    cases = [(768, 8192, 9, 512), (768, 8192, 50, 2), (256, 1000, 103, 64)]
    cases += [(16 * rng.randint(4, 64), int(2 ** rng.uniform(5, 15.7)), rng.randint(1, 200), rng.randint(1, 512))
              for _ in range(400)]
    for C, V, batch, P in cases:
        room, M = engine_workspace(C, V, batch, P), batch * P
        for rows, N, K in ((M, 3 * C, C), (M, C, C), (M, 4 * C, C), (M, C, 4 * C), (batch, V, C)):
            assert plan(rows, N, K, 1).ws_elems <= room, (C, V, batch, P, rows, N, K)


def test_row_strides_beyond_32_bit_offsets_stay_on_fp32_tiles():
    far = 1 << 22
    assert plan(1000, 1000, 32, 0, ldb=far - 4).kind == SPLIT and plan(1000, 1000, 32, 0, ldb=far).kind == MFMA
    for bt in (0, 1):
        assert plan(130, 4096, 32, bt).kind == SPLIT and plan(130, 4096, 32, bt, lda=far).kind == MFMA
    assert plan(4096, 130, 32, 1, ldb=far).kind == MFMA
    assert plan(65, far, 16, 0).kind == MFMA and plan(65, 64, far, 0).kind == MFMA and plan(65, 64, far, 1).kind == MFMA


def test_few_tiles_of_a_long_k_take_a_range_per_cu():
    """More than 16 K ranges, while there is a CU for each; what gemm_ex plans stays within its 16 MiB."""
    for bt in (0, 1):
        assert plan(128, 64, 65536, bt).splits >= 48 and plan(256, 128, 65536, bt).splits == 32
        assert plan(1024, 768, 50304, bt).splits <= 16 and plan(512, 512, 65536, bt).splits <= 16
        for M, N in ((65, 64), (65, 384), (256, 192), (300, 300), (128, 1000)):
            for K in (2048, 8192, 16384, 50304, 131072):
                p, tiles = plan(M, N, K, bt), -(-M // 64) * -(-N // 64)
                assert p.kind != SPLIT or p.splits <= 16 or (tiles * p.splits <= 256 and K >= 512 * p.splits), (M, N, K, p)
                assert p.ws_elems <= 4 << 20


def _packed_planes(mode, M, N, K, planes):
    l = {fh.NONE: K, fh.RIGHT: K, fh.LEFT: M}[mode], 1
    r = {fh.NONE: N, fh.RIGHT: K, fh.LEFT: N}[mode], 1
    return strided_tile(mode, M, N, K, *l, *r, N, 1, planes, M * K, N * K)


def test_large_strided_tiles_only_where_they_are_filled():
    for mode in (fh.NONE, fh.RIGHT, fh.LEFT):
        for M, N in ((64, 64), (16, 64), (24, 256), (100, 48), (192, 64), (130, 120)):
            assert _packed_planes(mode, M, N, 64, 2048) == 64, (M, N)
        assert _packed_planes(mode, 1024, 1024, 64, 12) == 128 and _packed_planes(mode, 128, 128, 64, 1024) == 128
        assert _packed_planes(mode, 120, 252, 64, 1024) == 128 and _packed_planes(mode, 1024, 64, 1024, 12) == 64


def test_planes_of_a_quarter_tile_stay_on_the_vector_kernel():
    for mode in (fh.NONE, fh.RIGHT, fh.LEFT):
        assert _packed_planes(mode, 32, 32, 64, 1024) == 0 and _packed_planes(mode, 16, 20, 256, 2048) == 0
        assert _packed_planes(mode, 32, 32, 256, 256) == 64 and _packed_planes(mode, 32, 32, 32, 1024) == 64
        assert _packed_planes(mode, 36, 32, 64, 1024) == 64

"""Plans of the products, on the host (256 CUs where there is no device)."""
import random

from plans import MFMA, SPLIT, engine_workspace, plan


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

"""The launch shape that the matrix-core GEMM chooses (no GPU needed: the rule is host arithmetic, for 256 compute units before a
device is opened): every shape covers its product, and products where two shapes were measured get the faster one."""
import random

import pytest

from tests._parity import gemm_shape as shape

Q4, Q5, Q6 = 12, 13, 14


def test_every_shape_covers_its_product():
    rng = random.Random(11)
    for _ in range(4000):
        wtype, pair = rng.choice((Q4, Q5, Q6)), rng.randint(0, 1)
        rows, nb, n = int(2 ** rng.uniform(0, 17)), rng.randint(1, 60), int(2 ** rng.uniform(0, 12))
        s = shape(wtype, rows, 256 * nb, n, pair)
        m_tiles, per_wg = (n + 15) // 16, 64 if s["narrow"] or pair else 128
        assert 1 <= s["tiles"] <= 8 and (s["columns"] - 1) * s["tiles"] < m_tiles <= s["columns"] * s["tiles"]
        assert (s["row_wgs"] - 1) * per_wg < rows <= s["row_wgs"] * per_wg
        assert (s["runs"] - 1) * s["sb_run"] < nb <= s["runs"] * s["sb_run"] and s["runs"] <= 16
        assert s["runs"] == 1 or (rows % 4 == 0 and not pair and s["sb_run"] >= 4)
        assert s["taken"] in (0, 1) and s["ns"] > 0


# us of the product with its quantizer, SwiGLU pass and planes: the shape that is wanted | the one an earlier estimate took
@pytest.mark.parametrize("wtype,rows,cols,n,want", [
    (Q4, 14336, 1024, 256, (1, 1, 8)),    # 17.6 | 18.7 (128 rows, four tiles)
    (Q4, 12288, 1024, 256, (1, 1, 8)),    # 17.3 | 18.4 (128 rows, four tiles)
    (Q4, 14336, 4096, 65, (1, 2, 5)),     # 24.8 | 26.6 (128 rows, four runs)
    (Q4, 4096, 14336, 96, (1, 8, 6)),     # 28.3 | 30.1 (128 rows, three tiles)
    (Q5, 12288, 1024, 200, (1, 1, 8)),    # 16.5 | 20.1 (128 rows, three tiles)
    (Q5, 16384, 1024, 256, (1, 1, 8)),    # 20.3 | 22.8 (128 rows, four tiles)
    (Q5, 6152, 2048, 65, (1, 1, 3)),      # 16.0 | 19.6 (128 rows, one tile)
    (Q5, 6152, 4096, 1000, (0, 1, 7)),    # 82.8 | 89.3 (eight tiles)
])
def test_single_products_take_the_faster_shape(wtype, rows, cols, n, want):
    s = shape(wtype, rows, cols, n)
    assert (s["narrow"], s["runs"], s["tiles"]) == want


@pytest.mark.parametrize("wtype,rows,cols,n,tiles", [
    (Q4, 4608, 1536, 391, 4),     # 27.5 | 42.1 (two launches)
    (Q4, 5632, 2048, 700, 8),     # 58.1 | 72.8 (two launches)
    (Q4, 10240, 5120, 391, 8),    # 106 | 135 (two launches)
    (Q4, 14336, 5120, 391, 8),    # 144 | 172 (two launches)
    (Q4, 11008, 4096, 200, 8),    # 64 | 74 (three tiles)
])
def test_pairs_take_the_faster_shape(wtype, rows, cols, n, tiles):
    s = shape(wtype, rows, cols, n, 1)
    assert s["taken"] == 1 and s["tiles"] == tiles


@pytest.mark.parametrize("rows,cols", [(2048, 1024), (4096, 4096), (5632, 2048), (11008, 4096), (10240, 5120), (14336, 4096)])
def test_one_more_row_changes_little(rows, cols):
    """No width where the pair's time jumps: one more activation row costs at most one more tile per workgroup."""
    before = shape(Q4, rows, cols, 64, 1)["ns"]
    for n in range(65, 1200):
        now = shape(Q4, rows, cols, n, 1)["ns"]
        assert now <= 1.35 * before, n
        before = now


@pytest.mark.parametrize("wtype,rows,cols,n", [(Q5, 10496, 4608, 17), (Q5, 9472, 4608, 68), (Q6, 8960, 4352, 101), (Q5, 10752, 5120, 29)])
def test_an_ffn_counts_the_quantizer_that_the_pair_adds(wtype, rows, cols, n):
    """Whole FFN with two launches | with the pair launch: 56.0 | 61.0, 70.5 | 76.2, 80.0 | 86.2, 57.3 | 62.2 us."""
    assert shape(wtype, rows, cols, n, 2)["taken"] == 0
    assert shape(wtype, rows, cols, 700, 2)["taken"] == 1


@pytest.mark.parametrize("wtype,n", [(Q4, 42), (Q5, 38), (Q5, 134), (Q6, 97), (Q6, 139)])
def test_few_rows_of_a_long_k_take_two_launches(wtype, n):
    """Gate and up of 4096 x 14336: two launches with K in runs against the one that cannot split it, 44.0 | 62.3, 48.6 | 89.4,
    86.5 | 115.7, 67.8 | 104.7, 83.4 | 114.6 us."""
    assert shape(wtype, 4096, 14336, n, 1)["taken"] == 0


@pytest.mark.parametrize("wtype,rows,cols,n", [(Q4, 513, 14336, 100), (Q5, 513, 14336, 100), (Q6, 513, 14336, 100), (Q5, 389, 10240, 79), (Q4, 283, 7936, 472),
                                               (Q5, 287, 12032, 476), (Q4, 915, 12032, 306)])
def test_few_ragged_rows_of_a_long_k_take_two_launches(wtype, rows, cols, n):
    """Gate and up of rows that do not divide by four: their two launches have K in runs over the padded rows.  Two launches | one, us:
    35.8 | 70.4, 38.1 | 99.1, 37.3 | 98.2, 29.9 | 63.0, 37.0 | 61.3, 44.7 | 111.2, 50.3 | 74.9."""
    assert shape(wtype, rows, cols, n, 1)["taken"] == 0


@pytest.mark.parametrize("wtype,rows,cols,n", [(Q4, 5633, 2048, 300), (Q4, 2047, 4096, 100), (Q5, 5605, 1536, 648), (Q6, 7587, 4096, 150), (Q4, 577, 3072, 67)])
def test_ragged_pairs_of_a_short_k_stay_in_one_launch(wtype, rows, cols, n):
    """One launch | two, us: 33.0 | 42.0, 27.5 | 29.9, 49.6 | 60.4, 47.5 | 59.5, 19.4 | 23.1."""
    assert shape(wtype, rows, cols, n, 1)["taken"] == 1

"""Which kernel a dense product takes (no GPU needed: the rule is host arithmetic, for 256 compute units before a device is opened)."""
import random

from tests._parity import PASSES, SIXTEENS, GEMM, dense_path


def products(count, seed):
    rng = random.Random(seed)
    for _ in range(count):
        yield rng.choice((12, 13, 14)), int(2 ** rng.uniform(4, 17)), rng.randint(1, 64), rng.randint(0, 1)


def test_up_to_sixteen_rows_stay_on_the_decode_kernels():
    for wtype, rows, nb, pair in products(20000, 5):
        assert dense_path(wtype, rows, nb, 8, pair)[0] == PASSES
        for n in (9, 16):
            path, _, sixteens = dense_path(wtype, rows, nb, n, pair)
            assert path == PASSES or (path == SIXTEENS and sixteens), (wtype, rows, nb, n, pair)
        assert dense_path(wtype, rows, nb, 65, pair)[0] == GEMM


def test_short_rows_and_pairs_of_ordinary_matrices_stay_on_the_decode_kernels_up_to_47_rows():
    """Of fewer than 44 million weights (24 MB of Q4_K): rows of up to 1024 columns, and gate/up pairs of any."""
    rng = random.Random(8)
    for _ in range(20000):
        wtype, pair, n = rng.choice((12, 13, 14)), rng.randint(0, 1), rng.randint(17, 47)
        nb = rng.randint(1, 64 if pair else 4)
        rows = int(2 ** rng.uniform(4, 15.4)) if not pair else rng.randint(1, (24 << 20) // (144 * nb))
        if rows * nb * 144 < 24 << 20:
            assert dense_path(wtype, rows, nb, n, pair)[0] != GEMM, (wtype, rows, nb, n, pair)


def test_tiles_of_sixteen_split_a_row_like_the_passes():
    for wtype, rows, nb, pair in products(20000, 6):
        for n in (9, 16, 17, 33, 64):
            path, passes, sixteens = dense_path(wtype, rows, nb, n, pair)
            assert sixteens in (0, passes) and (path != SIXTEENS or sixteens), (wtype, rows, nb, n, pair)


def test_down_product_behind_a_gemm_takes_the_faster_kernel():
    """Alone it stays with the tiles of sixteen unless the GEMM is far ahead; behind gate and up on the GEMM it need not."""
    for wtype, hidden, inter, n in ((14, 5120, 9216, 20), (12, 6144, 9472, 23), (13, 6144, 8704, 24), (12, 3840, 512, 54)):
        assert dense_path(wtype, hidden, inter // 256, n)[0] == SIXTEENS
        assert dense_path(wtype, hidden, inter // 256, n, 2)[0] == GEMM
    for wtype, hidden, inter, n in ((13, 3072, 2816, 48), (14, 2816, 2048, 49), (12, 1536, 2048, 53)):
        assert dense_path(wtype, hidden, inter // 256, n)[0] == dense_path(wtype, hidden, inter // 256, n, 2)[0] == SIXTEENS


def test_q80_rule_has_no_single_widths():
    """The row count from which the GEMM takes a Q8_0 product, over row lengths that the passes split over one wavefront count (eight, and
    four of more than 128 row tiles): longer rows keep it waiting, none of them alone."""
    def first(rows, nb):
        return next(n for n in range(1, 100) if dense_path(8, rows, nb, n)[0] == GEMM)
    for rows in (200, 700, 1041, 2000, 3328, 4096, 5000, 9000):
        for lengths in (range(8, 72, 8), range(36, 68, 8)):
            firsts = [first(rows, nb) for nb in lengths]
            assert firsts == sorted(firsts) and firsts[0] > 8, (rows, list(lengths), firsts)


def test_q80_up_to_eight_rows_are_passes_and_many_are_not():
    rng = random.Random(7)
    for _ in range(20000):
        rows, nb, n = int(2 ** rng.uniform(4, 17)), rng.randint(1, 64), rng.randint(1, 8)
        assert dense_path(8, rows, nb, n)[0] == PASSES, (rows, nb, n)
        assert dense_path(8, rows, nb, 64)[0] == (GEMM if rows * nb * 256 * 64 >= 1 << 21 else PASSES), (rows, nb)

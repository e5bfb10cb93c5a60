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


def test_tiles_of_sixteen_split_a_row_like_the_passes():
    for wtype, rows, nb, pair in products(20000, 6):
        for n in (9, 16, 17, 33, 64):
            path, passes, sixteens = dense_path(wtype, rows, nb, n, pair)
            assert sixteens in (0, passes) and (path != SIXTEENS or sixteens), (wtype, rows, nb, n, pair)

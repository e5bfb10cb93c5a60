"""Which kernel a dense product takes (no GPU needed: the rule is host arithmetic, for 256 compute units before a device is opened)."""
import ctypes as C
import random

from densecore_amd import _lib

PASSES, SIXTEENS, GEMM = 0, 1, 2


def dense_path(wtype, rows, nb, n, pair=0):
    out = (C.c_int * 3)()
    assert _lib.load().mq_debug_dense_path(wtype, rows, 256 * nb, n, pair, out) == 0
    return tuple(out)


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

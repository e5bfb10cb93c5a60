"""Shared helpers for the GPU parity tests."""
import numpy as np

from oracle import binding as orc

REL_TOL = 1e-4          # the path's stated fp32 bound (accumulation order only)
CANCEL_FLOOR = 1 / 64   # outputs smaller than this fraction of their summed term magnitudes are
                        # judged against that fraction instead (cancellation makes |ref| arbitrarily small)


def assert_fp32_parity(got: np.ndarray, ref: np.ndarray, mag: np.ndarray, what: str = "") -> float:
    """|got - ref| <= 1e-4 * max(|ref|, mag/64) element-wise; returns the largest plain relative
    error over the well-conditioned outputs (|ref| >= mag/64) for reporting."""
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    mag = np.asarray(mag, np.float64)
    assert got.shape == ref.shape, (got.shape, ref.shape)
    assert np.all(np.isfinite(got)), f"{what}: non-finite output"
    err = np.abs(got - ref)
    scale = np.maximum(np.abs(ref), mag * CANCEL_FLOOR)
    worst = np.max(err / np.maximum(scale, 1e-300))
    assert worst <= REL_TOL, f"{what}: max relative error {worst:.3e} > {REL_TOL}"
    ok = np.abs(ref) >= mag * CANCEL_FLOOR
    ok &= ref != 0          # ref == mag == 0 (an all-zero row): nothing to divide by
    return float(np.max(err[ok] / np.abs(ref[ok]))) if ok.any() else 0.0


def gemm_shape(wtype: int, rows: int, cols: int, n: int, pair: int = 0) -> dict:
    """The launch shape that the matrix-core GEMM chooses for a product (include/mi355_q4k_debug.h)."""
    import ctypes as C

    from densecore_amd import _lib
    out = (C.c_int * 8)()
    assert _lib.load().mq_debug_gemm_shape(wtype, rows, cols, n, pair, out) == 0
    return dict(zip(("narrow", "runs", "sb_run", "tiles", "row_wgs", "columns", "taken", "ns"), out))


def gemm_launch(wtype: int, rows: int, cols: int, n: int) -> dict:
    """The shape in which a GEMM product is launched: rows padded to four where that is the shorter one, Q8_0 included."""
    import ctypes as C

    from densecore_amd import _lib
    out = (C.c_int * 6)()
    assert _lib.load().mq_debug_gemm_launch(wtype, rows, cols, n, out) == 0
    return dict(zip(("narrow", "runs", "sb_run", "tiles", "row_wgs", "columns"), out))


PASSES, SIXTEENS, GEMM = 0, 1, 2


def dense_path(wtype: int, rows: int, nb: int, n: int, pair: int = 0) -> tuple:
    """Kernel of a dense product, wavefronts per row tile of the passes and of the tiles of sixteen (include/mi355_q4k_debug.h)."""
    import ctypes as C

    from densecore_amd import _lib
    out = (C.c_int * 3)()
    assert _lib.load().mq_debug_dense_path(wtype, rows, 256 * nb, n, pair, out) == 0
    return tuple(out)


def moe_path(gate_type: int, down_type: int, experts: int, hidden: int, inter: int, n: int, top_k: int) -> dict:
    """Whether gate/up and down of the layer, and the two nodes, run on the expert-grouped GEMM (include/mi355_q4k_debug.h)."""
    import ctypes as C

    from densecore_amd import _lib
    out = (C.c_int * 4)()
    assert _lib.load().mq_debug_moe_path(gate_type, down_type, experts, hidden, inter, n, top_k, out) == 0
    return dict(zip(("layer gateup", "layer down", "gateup", "down"), out))


def oracle_all_orders(w: np.ndarray, cols: int, q8: np.ndarray):
    return {name: orc.mul_mat_q4k_q8k(w, cols, q8, order) for name, order in orc.ORDERS.items()}

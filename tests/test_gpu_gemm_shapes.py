"""Launch shapes of the matrix-core GEMM: 64- and 128-row workgroups, activation tiles dealt over the workgroup columns, K in
runs.  The shapes sit where one of them changes; the reference is the oracle on sampled rows and the decode kernels on all."""
import numpy as np
import pytest

from densecore_amd import synth
from oracle import binding as orc
from tests._parity import assert_fp32_parity, gemm_shape

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


MAKE = {12: (synth.q4k_matrix, lambda *a: orc.mul_mat_q4k_q8k(*a, orc.ORDER_SCALAR), orc.dot_magnitude_f64),
        13: (synth.q5k_matrix, orc.mul_mat_q5k_q8k, lambda *a: orc.q5k_dot_dequant_f64(*a, magnitude=True)),
        14: (synth.q6k_matrix, orc.mul_mat_q6k_q8k, lambda *a: orc.q6k_dot_dequant_f64(*a, magnitude=True))}


# (narrow, runs, super-blocks per run, tiles per workgroup, columns) on 256 compute units
@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n,form", [
    (16, 256, 65, (1, 1, 1, 1, 5)), (20, 1024, 129, (1, 1, 4, 2, 5)),  # one workgroup row; a last column of one tile
    (1000, 3584, 145, (1, 3, 5, 2, 5)),      # 64 rows, 14 super-blocks as 5 + 5 + 4
    (4098, 3584, 391, (1, 1, 14, 4, 7)),     # rows that do not divide by four: no runs
    (2050, 4096, 260, (1, 1, 16, 3, 6)),     # 64 rows, ragged rows, 17 tiles dealt in threes
    (9000, 512, 400, (1, 1, 2, 8, 4)),       # a short K, in eights with a last column of one tile
    (14336, 1024, 512, (0, 1, 4, 8, 4)),     # 128 rows
    (13000, 1024, 505, (0, 1, 4, 7, 5)),     # 128 rows, ragged rows, 32 tiles as 7 + 7 + 7 + 7 + 4
    (4096, 14336, 130, {14: (1, 4, 14, 5, 2), 0: (0, 8, 7, 5, 2)}),  # K in runs over 128 rows (Q6_K: 64), nine tiles as 5 + 4
    (4096, 14336, 330, {13: (0, 8, 7, 7, 3), 14: (1, 5, 12, 7, 3), 0: (0, 5, 12, 7, 3)}),  # ... 56 super-blocks as 12 x 4 + 8
    (4096, 14336, 391, (0, 4, 14, 7, 4))])   # ... 25 tiles as 7 + 7 + 7 + 4, all three types over 128 rows
def test_gemm_shape(ops, wtype, rows, cols, n, form):
    import torch
    make, product, magnitude = MAKE[wtype]
    w = make(synth.tensor_seed("gs-w", rows, cols), rows, cols)
    x = synth.normal_f32(synth.tensor_seed("gs-x", n, cols), (n, cols))
    W = ops.Q4KWeight.from_ggml(w, cols, wtype)
    s = gemm_shape(wtype, rows, cols, n)
    if isinstance(form, dict):
        form = form.get(wtype, form[0])
    assert tuple(s[name] for name in ("narrow", "runs", "sb_run", "tiles", "columns")) == form, s
    xd = torch.from_numpy(x).cuda()
    yp = torch.full((n, rows + 8), 7.0, device="cuda")  # a padded output keeps its padding
    ops.gemm(W, xd, out=yp[:, :rows])
    assert bool((yp[:, rows:] == 7.0).all())
    got = yp[:, :rows]
    small = torch.cat([ops.mul_mat(W, xd[i:i + 8]) for i in range(0, n, 8)])
    assert (got - small).abs().max().item() <= 1e-5 * small.abs().max().item()  # same integers, fp32 summation order
    pick = np.unique(np.r_[0:rows:max(1, rows // 16), rows - 1])
    toks = np.unique(np.r_[0:n:max(1, n // 40), n - 1])
    q8 = orc.quantize_rows_q8k(x[toks])
    assert_fp32_parity(got.cpu().numpy()[np.ix_(toks, pick)], product(w[pick], cols, q8), magnitude(w[pick], cols, q8), "launch shape")
    W.free()


@pytest.mark.parametrize("rows,n,tiles", [(2064, 65, 1), (2064, 129, 2), (2064, 144, 2), (2064, 393, 4), (5648, 391, 5), (11008, 330, 5), (2064, 700, 7), (11008, 200, 8), (14336, 330, 8)])
def test_pair_launch_columns(ops, rows, n, tiles):
    """Gate and up in one launch: tiles dealt evenly, and in eights with a short last column (thirteen as 8 + 5, 21 as 8 + 8 + 5).
    No K runs at 1024 columns, so the two launches and the SwiGLU pass give the same bits."""
    import torch
    from densecore_amd import _lib
    s = gemm_shape(12, rows, 1024, n, 1)
    assert s["taken"] == 1 and s["tiles"] == tiles and gemm_shape(12, rows, 1024, n)["runs"] == 1
    G, U = (ops.Q4KWeight.synthetic(synth.tensor_seed("gs-p", t), rows, 1024) for t in "gu")
    x = torch.from_numpy(synth.normal_f32(synth.tensor_seed("gs-px", n), (n, 1024))).cuda()
    try:
        _lib.lib().mq_debug_set_dense_lds(1)
        h1 = ops.swiglu_mul_mat(G, U, x, ops.SILU_FAST)
        _lib.lib().mq_debug_set_dense_lds(1 | 8)
        h0 = ops.swiglu_mul_mat(G, U, x, ops.SILU_FAST)
    finally:
        _lib.lib().mq_debug_set_dense_lds(1)
    assert torch.equal(h1, h0)
    G.free(), U.free()

"""Launch shapes of the matrix-core GEMM: 64- and 128-row workgroups, activation tiles dealt over the workgroup columns, K in
runs.  The shapes sit where one of them changes; the reference is the oracle on sampled rows and the decode kernels on all."""
import numpy as np
import pytest

from densecore_amd import synth
from oracle import binding as orc
from tests._parity import assert_fp32_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


@pytest.mark.parametrize("rows,cols,n", [
    (16, 256, 65), (20, 1024, 129),          # one workgroup row; a second column of one tile
    (1000, 2048, 140), (1000, 2048, 145),    # nine tiles dealt 5 + 4, ten dealt 5 + 5
    (4104, 3584, 391), (4098, 3584, 391),    # K in runs over 128-row workgroups; rows that do not divide by four: no runs
    (2050, 4096, 260),                       # 64-row workgroups, ragged rows
    (9000, 512, 400)])                       # a short K: no runs
def test_gemm_shape(ops, rows, cols, n):
    import torch
    w = synth.q4k_matrix(synth.tensor_seed("gs-w", rows, cols), rows, cols)
    x = synth.normal_f32(synth.tensor_seed("gs-x", n, cols), (n, cols))
    W = ops.Q4KWeight.from_ggml(w, cols)
    xd = torch.from_numpy(x).cuda()
    yp = torch.full((n, rows + 8), 7.0, device="cuda")  # a padded output keeps its padding
    ops.gemm(W, xd, out=yp[:, :rows])
    assert bool((yp[:, rows:] == 7.0).all())
    got = yp[:, :rows]
    small = torch.cat([ops.mul_mat(W, xd[i:i + 8]) for i in range(0, n, 8)])
    assert (got - small).abs().max().item() <= 1e-5 * small.abs().max().item()  # same integers, fp32 summation order
    pick = np.unique(np.r_[0:rows:max(1, rows // 16), rows - 1])
    q8 = orc.quantize_rows_q8k(x)
    assert_fp32_parity(got.cpu().numpy()[:, pick], orc.mul_mat_q4k_q8k(w[pick], cols, q8, orc.ORDER_SCALAR),
                       orc.dot_magnitude_f64(w[pick], cols, q8), "launch shape")
    W.free()


@pytest.mark.parametrize("n", [65, 80, 129, 144, 384, 393])
def test_pair_launch_columns(ops, n):
    """Gate and up in one launch: five to 24 tiles dealt evenly, 25 in eights with a short column.  No K runs at 1024
    columns, so the two launches and the SwiGLU pass give the same bits."""
    import torch
    from densecore_amd import _lib
    G, U = (ops.Q4KWeight.synthetic(synth.tensor_seed("gs-p", t), 2064, 1024) for t in "gu")
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

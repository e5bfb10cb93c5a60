"""Q5_K and Q6_K on the matrix-core GEMM as two chains of byte digits: the forms they share with Q4_K (128-row workgroups,
gate and up in one launch, items of two, four and eight activation tiles)."""
import numpy as np
import pytest

from densecore_amd import synth
from oracle import binding as orc
from tests._parity import assert_fp32_parity, gemm_shape

pytestmark = pytest.mark.gpu
Q5, Q6 = synth.GGML_TYPE_Q5_K, synth.GGML_TYPE_Q6_K


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


def cu(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("wtype", [Q5, Q6])
def test_wide_workgroups_match_the_oracle(ops, wtype):
    """813 row tiles and 32 activation tiles: more 128-row workgroups than compute units, the last of each side ragged.
    Tokens of the first and the last activation tile against the oracle, all of them against the decode kernels
    (summation order only: the bound of assert_fp32_parity)."""
    import torch
    rows, cols, n = 13000, 1024, 505
    assert gemm_shape(wtype, rows, cols, n)["narrow"] == 0
    make, product, dequant = ((synth.q5k_matrix, orc.mul_mat_q5k_q8k, orc.q5k_dot_dequant_f64) if wtype == Q5 else
                              (synth.q6k_matrix, orc.mul_mat_q6k_q8k, orc.q6k_dot_dequant_f64))
    w = make(synth.tensor_seed("wd-w", wtype), rows, cols)
    x = synth.normal_f32(synth.tensor_seed("wd-x", wtype), (n, cols))
    W = ops.Q4KWeight.from_ggml(w, cols, wtype)
    got = ops.gemm(W, cu(x))
    small = torch.cat([ops.mul_mat(W, cu(x[i:i + 8])) for i in range(0, n, 8)])
    assert (got - small).abs().max().item() <= 1e-5 * small.abs().max().item()
    pick = np.r_[0:8, n - 8:n]
    q8 = orc.quantize_rows_q8k(x[pick])
    assert_fp32_parity(got.cpu().numpy()[pick], product(w, cols, q8), dequant(w, cols, q8, magnitude=True), "128-row workgroups")
    W.free()


@pytest.mark.parametrize("wtype", [Q5, Q6])
@pytest.mark.parametrize("n", [130, 1000])
def test_pair_launch_gives_the_bits_of_two_launches(ops, wtype, n):
    from densecore_amd import _lib
    hidden, inter = 1024, 2576
    G = ops.Q4KWeight.synthetic(synth.tensor_seed("wd-g", wtype), inter, hidden, 1, wtype)
    U = ops.Q4KWeight.synthetic(synth.tensor_seed("wd-u", wtype), inter, hidden, 1, wtype)
    x = cu(synth.normal_f32(synth.tensor_seed("wd-px", n), (n, hidden)))
    try:
        _lib.lib().mq_debug_set_dense_lds(1)
        h1 = ops.swiglu_mul_mat(G, U, x, ops.SILU_FAST).cpu().numpy()
        _lib.lib().mq_debug_set_dense_lds(1 | 8)
        h0 = ops.swiglu_mul_mat(G, U, x, ops.SILU_FAST).cpu().numpy()
    finally:
        _lib.lib().mq_debug_set_dense_lds(1)
    assert np.array_equal(h1.view(np.uint32), h0.view(np.uint32))
    G.free(), U.free()


@pytest.mark.parametrize("wtype", [Q5, Q6])
def test_items_and_pair_of_the_moe_block_give_the_same_bits(ops, wtype):
    """Items of two, four and eight tiles, gate and up in one launch or two (two tiles of Q5_K: the third chain)."""
    from densecore_amd import _lib
    n, E, H, I, K = 300, 12, 512, 256, 4
    ge, ue = (ops.Q4KWeight.synthetic(synth.tensor_seed("wd-m", t, wtype), I, H, E, wtype) for t in "gu")
    de = ops.Q4KWeight.synthetic(synth.tensor_seed("wd-m", "d", wtype), H, I, E, wtype)
    x = cu(synth.normal_f32(synth.tensor_seed("wd-mx"), (n, H)))
    lg = cu(synth.normal_f32(synth.tensor_seed("wd-ml"), (n, E)))
    out = []
    try:
        for mode in (1, 1 | (2 << 8), 1 | (4 << 8), 1 | (8 << 8), 9 | (2 << 8), 9 | (4 << 8), 9 | (8 << 8)):
            _lib.lib().mq_debug_set_dense_lds(mode)
            out.append(ops.moe_layer(ge, ue, de, x, lg, K, silu=ops.SILU_FAST)[0].cpu().numpy())
    finally:
        _lib.lib().mq_debug_set_dense_lds(1)
    for y in out[1:]:
        assert np.array_equal(y.view(np.uint32), out[0].view(np.uint32))
    for w in (ge, ue, de):
        w.free()


@pytest.mark.parametrize("scale,code", [(63, 31), (63, 0), (1, 31), (63, 2), (32, 4), (48, 8), (18, 21), (25, 5)])
def test_q5k_gemm_corners_of_the_byte_digits(ops, scale, code):
    """One scale and one code everywhere: the products scale * code = 1953, 0, 31 and those either side of a carry into the high
    byte (126 and 128, 378 and 384, 125), activations at +-full scale."""
    rows, cols, n = 32, 512, 70
    w_np = np.zeros((rows, cols // 256 * 176), np.uint8)
    blocks = w_np.reshape(rows, -1, 176)
    blocks[:, :, 0:2] = np.array([0.01], np.float16).view(np.uint8)
    blocks[:, :, 4:8] = scale | (scale >> 4) << 6   # scales 0..3, and the top bits of scales 4..7
    blocks[:, :, 12:16] = scale & 15                # mins stay zero
    blocks[:, :, 16:48] = 255 * (code >> 4)
    blocks[:, :, 48:176] = (code & 15) * 17
    x = np.ones((n, cols), np.float32)
    x[1::2] *= -1.0
    x[2, ::2] *= -1.0
    q8 = orc.quantize_rows_q8k(x)
    ds, md = orc.q5k_matrix_block_sums(w_np, cols, q8)
    assert np.all(np.abs(ds[:, 0]) == 127 * 256 * scale * code) and not md.any()
    W = ops.Q4KWeight.from_ggml(w_np, cols, Q5)
    got = ops.gemm(W, cu(x)).cpu().numpy()
    assert_fp32_parity(got, orc.mul_mat_q5k_q8k(w_np, cols, q8), orc.q5k_dot_dequant_f64(w_np, cols, q8, magnitude=True), "Q5_K corners")
    W.free()

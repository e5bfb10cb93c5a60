"""GPU: dense Q8_0 products of many rows (the GEMM over tiles of sixteen activation rows) against the launch of eight-row passes and,
where it is quick, the oracle.  Both form every 32-weight block's sum as an integer and add the scaled blocks of a row in fp32, in
another order: 1e-5 of the largest result covers the 2 K / 32 roundings of 2^-24 at the K used here.  Parity with the reference build
is unpinned (its activation quantizer is not in its tree)."""
import numpy as np
import pytest

from densecore_amd import synth
from oracle import binding as orc
from tests._parity import GEMM, assert_fp32_parity, dense_path

pytestmark = pytest.mark.gpu
Q80 = synth.GGML_TYPE_Q8_0


# one, two and four activation tiles to a workgroup, whole and partial last ones; whole and ragged row tiles; one and several super-blocks
@pytest.mark.parametrize("rows,cols,n,tiles", [(600, 256, 25, 1), (1000, 2048, 31, 1), (1003, 1792, 33, 1), (3072, 512, 17, 1), (8192, 256, 9, 1),
                                               (8200, 512, 63, 1), (8192, 256, 64, 1), (40, 1024, 512, 1), (16500, 512, 33, 2), (16500, 768, 48, 2),
                                               (16400, 512, 64, 2), (16500, 256, 129, 4), (2048, 768, 1030, 4)])
def test_many_rows_match_eight_at_a_time(rows, cols, n, tiles):
    import torch
    from densecore_amd import _lib, ops
    path, _, mt = dense_path(Q80, rows, cols // 256, n)
    assert (path, mt) == (GEMM, tiles)
    w = ops.Q4KWeight.synthetic(rows + n, rows, cols, 1, Q80)
    x = torch.randn(n, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    want = torch.cat([ops.mul_mat(w, x[i:i + 8]) for i in range(0, n, 8)])
    got = ops.mul_mat(w, x)
    assert (got - want).abs().max().item() <= 1e-5 * want.abs().max().item()
    apart = torch.full((n, cols + 20), float("nan"), device="cuda")  # rows 4 * 5 floats apart, not numbers between them
    apart[:, :cols] = x
    again = torch.empty_like(got)
    _lib.check(_lib.lib().mq_mul_mat_q4k(w._h, apart.data_ptr(), n, cols + 20, again.data_ptr(), rows, torch.cuda.current_stream().cuda_stream), "mq_mul_mat_q4k")
    assert torch.equal(got, again)
    w.free()


@pytest.mark.parametrize("rows,cols,n", [(96, 1024, 40), (35, 2560, 33)])
def test_many_rows_match_the_oracle(rows, cols, n):
    import torch
    from densecore_amd import ops
    w_np = synth.q80_matrix(synth.tensor_seed("mm80g-w", rows, cols), rows, cols)
    x = synth.normal_f32(synth.tensor_seed("mm80g-x", rows, cols, n), (n, cols))
    w = ops.Q4KWeight.from_ggml(w_np, cols, Q80)
    y = ops.mul_mat(w, torch.from_numpy(x).cuda()).cpu().numpy()
    q = orc.quantize_rows_q80(x, orc.Q80_X86)
    mag = orc.q80_dot_dequant_f64(w_np, cols, q, magnitude=True)
    assert_fp32_parity(y, orc.mul_mat_q80_q80(w_np, cols, q, orc.ORDER_HWY), mag, f"q80 gemm {rows}x{cols} n={n}")
    assert_fp32_parity(y, orc.q80_dot_dequant_f64(w_np, cols, q), mag, "q80 gemm vs double")
    w.free()


# the passes of eight split these rows over eight (4096, 14336 columns), five and four wavefronts; 14336 columns on more than one tile
# of rows, whose passes walk a row in one wavefront
@pytest.mark.parametrize("rows,cols,n", [(640, 4096, 40), (640, 14336, 40), (640, 5120, 64), (4200, 13312, 32), (8300, 14336, 16)])
def test_rounding_error_is_no_larger_than_that_of_eight_rows_at_a_time(rows, cols, n):
    """Both against the same quantized operands in double: the GEMM adds up super-blocks, the even and the odd ones apart, so that it does
    not lose to the passes' wavefronts (a plain chain over the row has up to 2.6 times their error)."""
    import torch
    from densecore_amd import ops
    w_np = synth.q80_matrix(synth.tensor_seed("mm80e-w", rows, cols), rows, cols)
    x = synth.normal_f32(synth.tensor_seed("mm80e-x", rows, cols, n), (n, cols))
    blk = w_np.reshape(rows, cols // 32, 34)
    scale = torch.from_numpy(blk[:, :, :2].copy().view(np.float16).astype(np.float64)).cuda()
    codes = torch.from_numpy(blk[:, :, 2:].copy().view(np.int8)).cuda().double()
    wd = (codes * scale).reshape(rows, cols)
    xb = x.reshape(n, cols // 32, 32)  # the quantizer of the library, in its own fp32 steps
    amax = np.abs(xb).max(-1, keepdims=True)
    xq = np.rint(xb * np.divide(np.float32(127), amax, where=amax != 0, out=np.zeros_like(amax)))
    xd = torch.from_numpy((xq.astype(np.float64) * (amax / np.float32(127)).astype(np.float16).astype(np.float64)).reshape(n, cols)).cuda()
    want = (xd @ wd.T.contiguous())
    w, xg = ops.Q4KWeight.from_ggml(w_np, cols, Q80), torch.from_numpy(x).cuda()
    error = lambda y: ((y.double() - want).norm() / want.norm()).item()
    gemm, passes = error(ops.mul_mat(w, xg)), error(torch.cat([ops.mul_mat(w, xg[i:i + 8]) for i in range(0, n, 8)]))
    assert passes < 1e-6  # the operands above are the library's
    assert gemm <= passes, (gemm, passes)
    w.free()

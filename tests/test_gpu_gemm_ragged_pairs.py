"""Gate and up of matrices whose rows do not divide by four, as two products with K in runs and as one launch."""
import pytest

from tests._parity import GEMM, dense_path, gemm_shape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n,one_launch", [(513, 14336, 100, 0), (389, 10240, 79, 0), (1, 8192, 65, 0), (1026, 12800, 257, 0), (2047, 2048, 130, 1)])
def test_ragged_pairs(wtype, rows, cols, n, one_launch):
    """Against the decode kernels: the same integers, fp32 sums of gate and up in another order -- 1e-5 of the largest |gate| |up|, their SiLU's slope
    being at most 1.1.  The padding of the output's rows stays as it was."""
    import torch
    from densecore_amd import _lib, ops
    assert dense_path(wtype, rows, cols // 256, n, 1)[0] == GEMM and gemm_shape(wtype, rows, cols, n, 1)["taken"] == one_launch
    G, U = (ops.Q4KWeight.synthetic(rows + s, rows, cols, 1, wtype) for s in (1, 2))
    x = torch.randn((n, cols), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    ld = (rows + 3) // 4 * 4 + 4

    def pair(start, count):
        h = torch.full((count, ld), 7.0, device="cuda")
        _lib.check(_lib.lib().mq_swiglu_mul_mat_q4k(G._h, U._h, x[start:].data_ptr(), count, cols, h.data_ptr(), ld, ops.SILU_FAST,
                                                    torch.cuda.current_stream().cuda_stream), "mq_swiglu_mul_mat_q4k")
        assert bool((h[:, rows:] == 7.0).all())
        return h[:, :rows]
    got, few = pair(0, n), torch.cat([pair(i, min(8, n - i)) for i in range(0, n, 8)])
    gate, up = (torch.cat([ops.mul_mat(w, x[i:i + 8]) for i in range(0, n, 8)]) for w in (G, U))
    assert bool(torch.isfinite(got).all())
    assert float((got - few).abs().max()) <= 2.2e-5 * float(gate.abs().max()) * float(up.abs().max())
    for w in (G, U):
        w.free()

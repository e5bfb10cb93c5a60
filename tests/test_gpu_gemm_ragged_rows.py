"""Matrices whose rows do not divide by four: K in runs over the rows padded to four, whose sums leave the padding out."""
import pytest

from tests._parity import gemm_launch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n", [(1, 4096, 65), (15, 4096, 70), (535, 12800, 108), (537, 8192, 66), (642, 8192, 130), (1023, 4096, 257),
                                         (2047, 5120, 391), (4097, 14336, 100), (4098, 14336, 67), (701, 2048, 100)])
def test_ragged_rows(ops, wtype, rows, cols, n):
    """Against the decode kernels: the same integers, another order of the fp32 sums; a padded output keeps its padding, the last row included."""
    import torch
    w = ops.Q4KWeight.synthetic(rows + n, rows, cols, 1, wtype)
    x = torch.randn((n, cols), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    launch = gemm_launch(wtype, rows, cols, n)
    assert launch["runs"] > 1 if cols > 2048 else launch["runs"] == (1 if wtype == 12 else 2)
    few = torch.cat([ops.mul_mat(w, x[i:i + 8].contiguous()) for i in range(0, n, 8)])
    wide = torch.full((n + 1, rows + 5), 7.0, device="cuda")
    for y, out in ((ops.gemm(w, x), None), (None, wide[:n, :rows])):
        if out is not None:
            y = ops.gemm(w, x, out=out)
            assert bool((wide[:n, rows:] == 7.0).all()) and bool((wide[n] == 7.0).all())
        assert bool(torch.isfinite(y).all())
        assert float((y - few).abs().max()) <= 1e-5 * float(few.abs().max())
    assert torch.equal(ops.mul_mat(w, x), ops.gemm(w, x))
    w.free()

"""The matrix-core GEMM's forms for five to eight activation tiles per workgroup, with whole and with short last columns."""
import pytest

from tests._parity import gemm_shape

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


# (rows, cols, tokens) -> (64-row workgroups, tiles per workgroup, tiles of the last column) for Q4_K; the other types take forms of their own
CASES = [(11024, 512, 391, (0, 5, 5)), (14352, 1024, 300, (0, 5, 4)), (8208, 512, 600, (0, 6, 2)), (14352, 1024, 448, (0, 7, 7)),
         (14352, 1024, 391, (0, 7, 4)), (14352, 512, 512, (0, 8, 8)), (14352, 1024, 330, (0, 8, 5)), (4112, 512, 240, (1, 5, 5)),
         (2064, 512, 500, (1, 5, 2)), (14352, 1024, 177, (1, 6, 6)), (2064, 512, 600, (1, 6, 2)), (8208, 512, 330, (1, 7, 7)),
         (5648, 512, 500, (1, 7, 4)), (11024, 512, 255, (1, 8, 8)), (5648, 512, 600, (1, 8, 6)), (2064, 256, 65, (1, 1, 1))]


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n,form", CASES)
def test_a_row_does_not_depend_on_the_form(ops, wtype, rows, cols, n, form):
    """K in one run: a token's results are one sequence of fp32 operations whatever tiles lie beside it, so they equal the launch over
    some of the tokens (other forms, other places in a tile) to the bit, and the decode kernels to the order of the sums."""
    import torch
    s = gemm_shape(wtype, rows, cols, n)
    assert s["runs"] == 1
    if wtype == 12:
        tiles = (n + 15) // 16
        assert (s["narrow"], s["tiles"], tiles - (s["columns"] - 1) * s["tiles"]) == form, s
    w = ops.Q4KWeight.synthetic(rows + n, rows, cols, 1, wtype)
    x = torch.randn((n, cols), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    y = ops.gemm(w, x)
    for start, count in ((0, 33), (max(0, n - 67), min(n, 67)), (n // 3, 48)):
        count = min(count, n - start)
        if gemm_shape(wtype, rows, cols, count)["runs"] == 1:
            assert torch.equal(y[start:start + count], ops.gemm(w, x[start:start + count].contiguous())), (start, count)
    for i in (0, n // 2 // 8 * 8, (n - 1) // 8 * 8):
        few = ops.mul_mat(w, x[i:i + 8].contiguous())
        assert float((y[i:i + 8] - few).abs().max()) <= 1e-5 * float(few.abs().max())  # same integers, fp32 summation order
    w.free()


# whole and short last columns of every form, and workgroups of fewer tiles than the form of five
@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n,tiles", [(5648, 512, 80, 3), (5648, 512, 96, 3), (5648, 512, 112, 4), (5648, 512, 128, 4), (5648, 512, 129, 5), (5648, 512, 177, 6),
                                               (5648, 512, 195, 7), (5648, 512, 255, 8), (5648, 512, 391, 5), (14336, 1024, 112, 7), (14336, 1024, 330, 8)])
def test_pair_rows_do_not_depend_on_the_form(ops, wtype, rows, cols, n, tiles):
    """gate and up in one launch: the rows of a prefix of the tokens, bit for bit (a pair has no runs)."""
    import torch
    shape = gemm_shape(wtype, rows, cols, n, 1)
    assert shape["taken"] and shape["tiles"] == tiles
    g, u = (ops.Q4KWeight.synthetic(s, rows, cols, 1, wtype) for s in (1, 2))
    x = torch.randn((n, cols), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    h = ops.swiglu_mul_mat(g, u, x, ops.SILU_FAST)
    for count in (66, n - 1):
        assert gemm_shape(wtype, rows, cols, count, 1)["taken"]
        assert torch.equal(h[:count], ops.swiglu_mul_mat(g, u, x[:count].contiguous(), ops.SILU_FAST)), count
    for w in (g, u):
        w.free()

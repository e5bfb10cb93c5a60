"""Dense products of nine to 64 rows where an estimate leaves the plain choice of kernel: long rows whose super-blocks one wavefront
would walk alone, rows a little beyond a pass of sixteen.  Against the same rows handed over eight at a time (the decode kernels, held
to the oracle elsewhere): the same integers, fp32 sums in another order, one fp32 rounding per super-block and product term."""
import pytest

pytestmark = pytest.mark.gpu


def pieces(torch, fn, x):
    return torch.cat([fn(x[i:i + 8]) for i in range(0, x.shape[0], 8)])


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,nb", [(512, 19), (516, 43), (1030, 29), (3323, 31), (4608, 7), (8190, 53), (40960, 13)])
def test_products_match_their_rows_eight_at_a_time(wtype, rows, nb):
    import torch
    from densecore_amd import ops
    w = ops.Q4KWeight.synthetic(rows * 64 + nb, rows, 256 * nb, 1, wtype)
    x = torch.randn((64, 256 * nb), device="cuda", generator=torch.Generator(device="cuda").manual_seed(nb))
    want = pieces(torch, lambda t: ops.mul_mat(w, t), x)
    for n in (9, 16, 17, 31, 33, 47, 48, 64):
        got = ops.mul_mat(w, x[:n])
        # nb <= 53 roundings of 2^-24 on either side, each at most the largest partial sum (a few times the largest result)
        assert (got - want[:n]).abs().max().item() <= 1e-5 * want.abs().max().item(), n
    w.free()


@pytest.mark.parametrize("wtype,down_type,hidden,inter", [(12, 12, 2560, 11008), (12, 14, 2816, 5888), (13, 12, 1280, 7424), (14, 13, 4864, 9984),
                                                           (13, 14, 5120, 9216), (13, 13, 3072, 2816)])
def test_ffn_with_each_product_on_its_own_kernel(wtype, down_type, hidden, inter):
    import torch
    from densecore_amd import ops
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, 1, wtype) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, 1, down_type)
    x = torch.randn((64, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(inter))
    want = pieces(torch, lambda t: ops.ffn_swiglu(G, U, D, t, ops.SILU_FAST_FMA), x)
    for n in (9, 20, 33, 40, 64):
        got = ops.ffn_swiglu(G, U, D, x[:n], ops.SILU_FAST_FMA)
        # behind the second quantizer a last-bit difference moves a code by one now and then: one of 127 in a few of the products
        assert ((got - want[:n]).norm() / want[:n].norm()).item() <= 2e-4, n
    for w in (G, U, D):
        w.free()

"""MoE blocks on either side of the line between the decode launches and the expert-grouped GEMM."""
import pytest

from tests._parity import moe_path

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


def near(got, want):
    # another order of sums now and then moves an 8-bit code of a hidden row by one: at most 1 / 254 of the row's largest value on one of
    # its 256, so 4e-3 of the outputs' scale and far less on average
    import torch
    scale = want.abs().max()
    assert float((got - want).abs().max()) <= 4e-3 * float(scale)
    assert float((got - want).double().pow(2).mean().sqrt()) <= 2e-4 * float(want.double().pow(2).mean().sqrt())
    assert bool(torch.isfinite(got).all())


# (tokens, experts, top_k, hidden, inter, on the GEMM): the fewest tokens with rows enough and one token less; the fewest pairs and fewer; rows per
# expert at the line (17 x 4 over 24 experts: 2.83 of 2.78 rows at inter 256) and below it; hidden rows in place and in tiles; few rows
# per expert at prefill width; items of four tiles, whole and short; nine and sixteen tokens with three super-blocks of a row and with
# seven to a wavefront, six rows per expert and fewer
@pytest.mark.parametrize("n,experts,k,hidden,inter,gemm", [(17, 8, 8, 512, 256, 1), (16, 8, 8, 512, 256, 0), (32, 4, 2, 512, 256, 1), (31, 4, 2, 512, 256, 0),
                                                           (17, 24, 4, 512, 256, 1), (17, 25, 4, 512, 256, 0), (64, 40, 4, 768, 512, 1), (65, 40, 4, 768, 512, 1),
                                                           (200, 200, 4, 512, 512, 1), (193, 256, 4, 512, 256, 1),
                                                           (200, 12, 4, 768, 512, 1), (131, 9, 4, 512, 768, 1), (333, 9, 2, 512, 256, 1),
                                                           (9, 8, 8, 2304, 512, 0), (9, 8, 8, 1792, 768, 1), (16, 10, 4, 1792, 512, 1), (16, 11, 4, 1792, 512, 0)])
@pytest.mark.parametrize("types", [("q4_k", "q4_k"), ("q6_k", "q5_k"), ("q5_k", "q6_k")])
def test_layer_is_its_nodes_and_agrees_with_one_token_at_a_time(ops, n, experts, k, hidden, inter, gemm, types):
    import torch
    T = {"q4_k": ops.GGML_TYPE_Q4_K, "q5_k": ops.GGML_TYPE_Q5_K, "q6_k": ops.GGML_TYPE_Q6_K}
    gu, dn = T[types[0]], T[types[1]]
    assert set(moe_path(gu, dn, experts, hidden, inter, n, k).values()) == {gemm}
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, experts, gu) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, experts, dn)
    sh = (ops.Q4KWeight.synthetic(4, inter, hidden, 1, gu), ops.Q4KWeight.synthetic(5, inter, hidden, 1, gu), ops.Q4KWeight.synthetic(6, hidden, inter, 1, dn))
    gen = torch.Generator(device="cuda").manual_seed(n + experts)
    x, lg = torch.randn((n, hidden), device="cuda", generator=gen), torch.randn((n, experts), device="cuda", generator=gen)
    gi = torch.randn(hidden, device="cuda", generator=gen) * hidden ** -0.5
    y, ids, w = ops.moe_layer(G, U, D, x, lg, k, silu=ops.SILU_FAST)
    h = ops.moe_gateup_swiglu(G, U, x, ids, ops.SILU_FAST)
    assert torch.equal(y, ops.moe_down_weighted(D, h, ids, w))
    if n <= 64:
        ops.moe_layer(G, U, D, x, lg, k, silu=ops.SILU_FAST)
        assert torch.equal(ops.debug_moe_hidden((n, k, inter)), h)
    ys, ids_s, _ = ops.moe_layer(G, U, D, x, lg, k, shared=(*sh, gi), silu=ops.SILU_FAST)
    assert torch.equal(ids_s, ids)
    pick = sorted({0, 1, n // 2, n - 1})
    for shared, full in ((None, y), ((*sh, gi), ys)):  # one token: the token-major launches
        one = torch.cat([ops.moe_layer(G, U, D, x[t:t + 1].contiguous(), lg[t:t + 1].contiguous(), k, shared=shared, silu=ops.SILU_FAST)[0] for t in pick])
        near(full[pick], one)
    for m in (G, U, D, *sh):
        m.free()


# one product each way: few experts whose gate/up product would lose on the GEMM, few pairs of long rows, a down product of several wavefronts
# a row; (gate/up, down) on the GEMM
@pytest.mark.parametrize("n,experts,k,hidden,inter,gemm", [(18, 16, 4, 3072, 256, (0, 1)), (50, 32, 2, 3072, 256, (0, 1)), (17, 8, 6, 4096, 512, (0, 1)), (27, 8, 2, 1280, 768, (1, 0)),
                                                           (25, 8, 2, 1280, 1024, (1, 0))])
@pytest.mark.parametrize("gu,dn", [(12, 12), (12, 14), (14, 13)])
def test_layer_of_one_product_each_way_is_its_nodes(ops, n, experts, k, hidden, inter, gemm, gu, dn):
    import torch
    p = moe_path(gu, dn, experts, hidden, inter, n, k)
    if gu == 12:
        assert (p["layer gateup"], p["layer down"]) == gemm
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, experts, gu) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, experts, dn)
    sh = (ops.Q4KWeight.synthetic(4, inter, hidden, 1, gu), ops.Q4KWeight.synthetic(5, inter, hidden, 1, gu), ops.Q4KWeight.synthetic(6, hidden, inter, 1, dn))
    gen = torch.Generator(device="cuda").manual_seed(n + experts)
    x, lg = torch.randn((n, hidden), device="cuda", generator=gen), torch.randn((n, experts), device="cuda", generator=gen)
    gi = torch.randn(hidden, device="cuda", generator=gen) * hidden ** -0.5
    y, ids, w = ops.moe_layer(G, U, D, x, lg, k, silu=ops.SILU_FAST)
    rows = ops.debug_moe_hidden((n, k, inter))
    h = ops.moe_gateup_swiglu(G, U, x, ids, ops.SILU_FAST)
    assert torch.equal(rows, h) and torch.equal(y, ops.moe_down_weighted(D, h, ids, w))
    ys = ops.moe_layer(G, U, D, x, lg, k, shared=(*sh, gi), silu=ops.SILU_FAST)[0]
    pick = sorted({0, 1, n // 2, n - 1})
    for shared, full in ((None, y), ((*sh, gi), ys)):
        one = torch.cat([ops.moe_layer(G, U, D, x[t:t + 1].contiguous(), lg[t:t + 1].contiguous(), k, shared=shared, silu=ops.SILU_FAST)[0] for t in pick])
        near(full[pick], one)
    for m in (G, U, D, *sh):
        m.free()

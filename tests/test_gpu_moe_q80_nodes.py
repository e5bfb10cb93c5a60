"""The gate/up node ahead of a Q8_0 down stack, on the decode launches and on the expert-grouped GEMM."""
import pytest

from tests._parity import moe_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gate,experts,k,hidden,inter,n,gateup,layer", [(13, 16, 4, 3072, 256, 18, 0, 0), (12, 8, 6, 4096, 512, 17, 0, 0), (14, 16, 8, 1024, 768, 30, 1, 0),
                                                                        (12, 8, 2, 1280, 768, 27, 1, 0), (13, 32, 4, 768, 256, 200, 1, 1)])
def test_nodes_and_layer_agree_with_one_token_at_a_time(gate, experts, k, hidden, inter, n, gateup, layer):
    """gate/up rows: the same integers, fp32 sums in another order; behind them an 8-bit code of a hidden row now and then moves by one,
    1 / 254 of the largest of its 32 values."""
    import torch
    from densecore_amd import ops
    p = moe_path(gate, 8, experts, hidden, inter, n, k)
    assert (p["gateup"], p["layer gateup"], p["down"]) == (gateup, layer, 0)
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, experts, gate) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, experts, 8)
    gen = torch.Generator(device="cuda").manual_seed(n)
    x, lg = torch.randn((n, hidden), device="cuda", generator=gen), torch.randn((n, experts), device="cuda", generator=gen)
    y, ids, w = ops.moe_layer(G, U, D, x, lg, k, silu=ops.SILU_FAST)
    h = ops.moe_gateup_swiglu(G, U, x, ids, ops.SILU_FAST)
    nodes = ops.moe_down_weighted(D, h, ids, w)
    if gateup == layer:
        assert torch.equal(y, nodes)
    pick = sorted({0, 1, n // 2, n - 1})
    one = [(ops.moe_gateup_swiglu(G, U, x[t:t + 1], ids[t:t + 1], ops.SILU_FAST), ops.moe_layer(G, U, D, x[t:t + 1], lg[t:t + 1], k, silu=ops.SILU_FAST)[0]) for t in pick]
    rows, want = (torch.cat([o[i].reshape(1, -1) for o in one]) for i in (0, 1))
    assert float((h[pick].reshape(len(pick), -1) - rows).abs().max()) <= 2e-5 * float(rows.abs().max())
    for got in (y, nodes):
        assert bool(torch.isfinite(got).all())
        assert float((got[pick] - want).abs().max()) <= 4e-3 * float(want.abs().max())
        assert float((got[pick] - want).double().pow(2).mean().sqrt()) <= 2e-4 * float(want.double().pow(2).mean().sqrt())
    for m in (G, U, D):
        m.free()

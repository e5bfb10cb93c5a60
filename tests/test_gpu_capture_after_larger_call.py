"""One eager call of the largest width, then smaller ones captured: whichever kernels a smaller width takes, its workspaces are there
(nothing can be allocated under capture), and the replays return the eager call's bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ops():
    """The library as a program finds it: no workspace allocated yet."""
    import torch
    from densecore_amd import _lib, ops as o
    torch.cuda.synchronize()
    _lib.check(_lib.lib().mq_shutdown(), "mq_shutdown")
    _lib.check(_lib.lib().mq_init(torch.cuda.current_device()), "mq_init")
    return o


def captured_equals_eager(call):
    """call(): one product into tensors of its own, returned as a tuple.  Captured before it has ever run eagerly."""
    import torch
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        got = call()
    graph.replay()
    torch.cuda.synchronize()
    first = [t.clone() for t in got]
    want = call()
    for _ in range(2):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b, c in zip(got, want, first):
            assert torch.equal(a, b) and torch.equal(c, b)


def moe_weights(ops, experts, hidden, inter, gate=12, down=12):
    return (ops.Q4KWeight.synthetic(1, inter, hidden, experts, gate), ops.Q4KWeight.synthetic(2, inter, hidden, experts, gate),
            ops.Q4KWeight.synthetic(3, hidden, inter, experts, down))


@pytest.mark.parametrize("experts,k,hidden,inter,shared,eager,n", [(16, 8, 1024, 768, False, 300, 48), (16, 4, 512, 512, True, 200, 64)])
def test_layer_with_its_rows_in_place(ops, experts, k, hidden, inter, shared, eager, n):
    """The eager call leaves its hidden rows in the GEMM's tiles; up to 64 tokens they lie at their (token, slot) places."""
    import torch
    G, U, D = moe_weights(ops, experts, hidden, inter)
    sh = None
    if shared:
        sh = (*moe_weights(ops, 1, hidden, inter), torch.randn(hidden, device="cuda") * hidden ** -0.5)
    x, lg = torch.randn((eager, hidden), device="cuda"), torch.randn((eager, experts), device="cuda")
    ops.moe_layer(G, U, D, x, lg, k, shared=sh, silu=ops.SILU_FAST)
    captured_equals_eager(lambda: ops.moe_layer(G, U, D, x[:n], lg[:n], k, shared=sh, silu=ops.SILU_FAST))
    for w in (G, U, D, *(sh or ())[:3]):
        w.free()


# blocks whose eager width takes the expert-grouped GEMM and whose captured ones take the decode launches; the other way round (rows per expert
# do not decide alone); a Q8_0 down stack; few experts of long rows, where nine tokens take the GEMM already
BLOCKS = [(64, 6, 512, 512, 12, True, 256, (1, 5, 9, 20, 30, 100)), (16, 8, 512, 256, 14, False, 64, (2, 8, 12, 16, 17, 40)),
          (8, 2, 512, 1024, 13, False, 96, (1, 9, 20, 31, 32, 64)), (32, 4, 512, 512, 8, True, 300, (3, 9, 24, 60, 200)),
          (8, 8, 2304, 256, 12, False, 40, (1, 8, 9, 16, 24))]


@pytest.mark.parametrize("experts,k,hidden,inter,down,shared,eager,widths", BLOCKS)
def test_layer_at_every_width(ops, experts, k, hidden, inter, down, shared, eager, widths):
    import torch
    G, U, D = moe_weights(ops, experts, hidden, inter, down=down)
    sh = None
    if shared:
        sh = (*moe_weights(ops, 1, hidden, inter, down=down), None)
    x, lg = torch.randn((eager, hidden), device="cuda"), torch.randn((eager, experts), device="cuda")
    ops.moe_layer(G, U, D, x, lg, k, shared=sh, silu=ops.SILU_FAST)
    for n in widths:
        captured_equals_eager(lambda: ops.moe_layer(G, U, D, x[:n], lg[:n], k, shared=sh, silu=ops.SILU_FAST))
    for w in (G, U, D, *(sh or ())[:3]):
        w.free()


@pytest.mark.parametrize("experts,k,hidden,inter,down,shared,eager,widths", BLOCKS)
@pytest.mark.parametrize("node", ["gate/up", "down", "product", "product of slot rows"])
def test_expert_nodes_at_every_width(ops, node, experts, k, hidden, inter, down, shared, eager, widths):
    import torch
    G, U, D = moe_weights(ops, experts, hidden, inter, down=down)
    x, lg = torch.randn((eager, hidden), device="cuda"), torch.randn((eager, experts), device="cuda")
    h, w = torch.randn((eager, k, inter), device="cuda"), torch.rand((eager, k), device="cuda")
    ids = torch.topk(lg, k, 1).indices.int().contiguous()
    xs = torch.randn((eager, k, hidden), device="cuda")
    call = {"gate/up": lambda n: ops.moe_gateup_swiglu(G, U, x[:n], ids[:n], ops.SILU_FAST),
            "down": lambda n: ops.moe_down_weighted(D, h[:n], ids[:n], w[:n]),
            "product": lambda n: ops.mul_mat_id(G, x[:n], ids[:n]),
            "product of slot rows": lambda n: ops.mul_mat_id(G, xs[:n], ids[:n])}[node]
    call(eager)
    for n in widths:
        captured_equals_eager(lambda: (call(n),))
    for m in (G, U, D):
        m.free()

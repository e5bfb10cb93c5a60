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
          (8, 8, 2304, 256, 12, False, 40, (1, 8, 9, 16, 24)), (16, 4, 3072, 256, 12, True, 400, (5, 18, 24, 100)), (8, 2, 1280, 768, 13, False, 200, (9, 25, 27, 31, 64))]


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


# K in runs at the captured width and whole at the eager one; every kernel of a dense product below
@pytest.mark.parametrize("wtype,rows,cols,eager,widths", [(12, 2000, 16384, 4096, (1, 3, 9, 17, 40, 65, 100, 700)), (12, 2001, 16384, 4096, (2, 33, 100)),
                                                          (13, 4096, 4096, 600, (1, 8, 16, 24, 50, 64, 100)), (14, 6144, 1024, 300, (4, 12, 33, 48, 70)),
                                                          (8, 2000, 16384, 4096, (1, 8, 9, 17, 40, 100)), (8, 16, 256, 3000, (1, 30, 100, 400))])
def test_product_at_every_width(ops, wtype, rows, cols, eager, widths):
    import torch
    w = ops.Q4KWeight.synthetic(rows, rows, cols, 1, wtype)
    x = torch.randn((eager, cols), device="cuda")
    ops.mul_mat(w, x)
    for n in widths:
        captured_equals_eager(lambda: (ops.mul_mat(w, x[:n]),))
    w.free()


@pytest.mark.parametrize("types,hidden,inter,eager,widths", [((12, 14), 1024, 4096, 1000, (1, 2, 5, 9, 13, 17, 33, 50, 64, 65, 130, 391)),
                                                             ((13, 12), 5120, 1024, 300, (1, 8, 16, 30, 64, 100)), ((14, 13), 768, 2816, 64, (1, 4, 12, 17, 40))])
def test_ffn_and_pair_at_every_width(ops, types, hidden, inter, eager, widths):
    import torch
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, 1, types[0]) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, 1, types[1])
    x = torch.randn((eager, hidden), device="cuda")
    ops.ffn_swiglu(G, U, D, x)
    for n in widths:
        captured_equals_eager(lambda: (ops.ffn_swiglu(G, U, D, x[:n]),))
    for m in (G, U, D):
        m.free()


@pytest.mark.parametrize("wtype,rows,cols,eager,widths", [(12, 4096, 14336, 400, (1, 9, 20, 42, 64, 100, 140)), (13, 513, 6144, 300, (3, 17, 50, 100))])
def test_pair_by_itself_at_every_width(ops, wtype, rows, cols, eager, widths):
    import torch
    G, U = (ops.Q4KWeight.synthetic(s, rows, cols, 1, wtype) for s in (1, 2))
    x = torch.randn((eager, cols), device="cuda")
    ops.swiglu_mul_mat(G, U, x, ops.SILU_FAST)
    for n in widths:
        captured_equals_eager(lambda: (ops.swiglu_mul_mat(G, U, x[:n], ops.SILU_FAST),))
    for m in (G, U):
        m.free()


@pytest.mark.parametrize("eager,widths", [(300, (1, 2, 5, 16, 20, 48, 64, 100))])
def test_norm_and_product_at_every_width(ops, eager, widths):
    import torch
    from densecore_amd import _lib
    rows, cols = 4096, 2560
    w = ops.Q4KWeight.synthetic(5, rows, cols)
    x, g = torch.randn((eager, cols), device="cuda"), torch.randn(cols, device="cuda")

    def call(n):
        y = torch.empty((n, rows), device="cuda")
        _lib.check(_lib.lib().mq_rmsnorm_mul_mat_q4k(w._h, x.data_ptr(), None, g.data_ptr(), n, 1e-6, None, y.data_ptr(), rows,
                                                     torch.cuda.current_stream().cuda_stream), "mq_rmsnorm_mul_mat_q4k")
        return (y,)
    call(eager)
    for n in widths:
        captured_equals_eager(lambda: call(n))
    w.free()

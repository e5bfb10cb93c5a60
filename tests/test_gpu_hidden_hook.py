"""mq_debug_moe_hidden hands out the rows of the last layer or FFN call, or an error where that call left none: never another call's."""
import pytest

pytestmark = pytest.mark.gpu


def test_rows_of_the_last_call_or_an_error():
    import torch
    from densecore_amd import _lib, ops
    experts, top_k, hidden, inter = 16, 8, 2816, 768
    gen = torch.Generator(device="cuda").manual_seed(3)
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, experts) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, experts)
    D8 = ops.Q4KWeight.synthetic(3, hidden, inter, experts, ops.GGML_TYPE_Q8_0)
    x, logits = torch.randn(256, hidden, device="cuda", generator=gen), torch.randn(256, experts, device="cuda", generator=gen)

    def layer(n, down=D):
        return ops.moe_layer(G, U, down, x[:n].contiguous(), logits[:n].contiguous(), top_k, silu=ops.SILU_FAST)[1]

    def rows(n, ids):
        return ops.moe_gateup_swiglu(G, U, x[:n].contiguous(), ids, ops.SILU_FAST)

    ids = layer(8)
    assert torch.equal(ops.debug_moe_hidden((8, top_k, inter)), rows(8, ids))
    with pytest.raises(_lib.MqError):  # more than the call left
        ops.debug_moe_hidden((9, top_k, inter))
    for n in (128, 256):  # the expert-grouped GEMM: the rows stay in its tiles
        layer(n)
        with pytest.raises(_lib.MqError):
            ops.debug_moe_hidden((n, top_k, inter))
    ids = layer(256, D8)  # ... unless the down stack takes them as fp32
    assert torch.equal(ops.debug_moe_hidden((256, top_k, inter)), rows(256, ids))

    dg, du = (ops.Q4KWeight.synthetic(s, 2048, 1024) for s in (4, 5))
    dd = ops.Q4KWeight.synthetic(6, 1024, 2048)
    for n in (1, 13, 50, 400):
        ops.ffn_swiglu(dg, du, dd, x[:1, :1024].expand(n, 1024).contiguous(), ops.SILU_FAST)
        got = ops.debug_moe_hidden((n, 2048))
        assert bool((got.abs().sum(1) > 0).all()) and torch.equal(got[0], got[n - 1])
    xn, yn = torch.randn(300, 1024, device="cuda", generator=gen), torch.empty(300, 2048, device="cuda")
    _lib.check(_lib.lib().mq_rmsnorm_mul_mat_q4k(dg._h, xn.data_ptr(), None, None, 300, 1e-6, None, yn.data_ptr(), 2048,
                                                 torch.cuda.current_stream().cuda_stream), "mq_rmsnorm_mul_mat_q4k")
    with pytest.raises(_lib.MqError):  # the normalised rows lie there now
        ops.debug_moe_hidden((300, 1024))
    for w in (G, U, D, D8, dg, du, dd):
        w.free()

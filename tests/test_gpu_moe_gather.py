"""Expert products at prefill widths, whose GEMM gathers its activation rows itself: row counts around the quantizer's four rows to a
workgroup and the sixteen-row tiles, experts with no, one and many rows, every item size, rows per token and per (token, slot)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("item_tiles", [2, 4, 8])
@pytest.mark.parametrize("wtype,n,x_slots", [(12, 192, 1), (12, 193, 3), (13, 194, 1), (13, 257, 3), (14, 195, 3), (14, 271, 1)])
def test_gathered_rows_match_the_decode_groups(wtype, n, x_slots, item_tiles):
    import torch
    from densecore_amd import _lib, ops
    experts, top_k, rows, cols = 7, 3, 84, 768
    w = ops.Q4KWeight.synthetic(31, rows, cols, experts, wtype)
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((n, cols) if x_slots == 1 else (n, top_k, cols), device="cuda", generator=gen)
    # expert 0 takes a slot of most tokens, expert 5 that of one token, expert 6 none; an id out of range is a row without a product
    ids = torch.randint(0, 5, (n, top_k), device="cuda", generator=gen, dtype=torch.int32)
    ids[n // 4:, 0] = 0
    ids[3, 1], ids[5, 2] = 5, -1
    _lib.lib().mq_debug_set_dense_lds(1 | item_tiles << 8)
    try:
        got = ops.mul_mat_id(w, x, ids)
    finally:
        _lib.lib().mq_debug_set_dense_lds(1)
    want = torch.cat([ops.mul_mat_id(w, x[i:i + 8].contiguous(), ids[i:i + 8].contiguous()) for i in range(0, n, 8)])
    assert bool((got[5, 2] == 0).all())
    # the same integers, fp32 sums over three super-blocks in another order: 3 x 2^-24 of the largest term, with a factor to spare
    assert (got - want).abs().max().item() <= 1e-5 * want.abs().max().item()
    w.free()


@pytest.mark.parametrize("item_tiles", [2, 4, 8])
@pytest.mark.parametrize("wtype,rows,cols", [(12, 84, 512), (12, 132, 256), (13, 256, 512), (13, 20, 1024), (14, 128, 512), (14, 276, 768)])
def test_down_rows_with_resident_activations_match_the_staged_ones(wtype, rows, cols, item_tiles):
    """One slot of weight one: the down product's row itself, from a workgroup that keeps all super-blocks of its rows (up to eight
    tiles and super-blocks, below and beyond 128 weight rows), against mul_mat_id, which stages one super-block at a time."""
    import torch
    from densecore_amd import _lib, ops
    experts, n = 5, 211
    w = ops.Q4KWeight.synthetic(47, rows, cols, experts, wtype)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((n, 1, cols), device="cuda", generator=gen)
    ids = torch.randint(0, experts - 1, (n, 1), device="cuda", generator=gen, dtype=torch.int32)
    ids[7], ids[9] = experts - 1, experts  # an expert with one row, an id without an expert
    _lib.lib().mq_debug_set_dense_lds(1 | item_tiles << 8)
    try:
        got = ops.moe_down_weighted(w, x, ids, torch.ones((n, 1), device="cuda"))
        want = ops.mul_mat_id(w, x, ids)
    finally:
        _lib.lib().mq_debug_set_dense_lds(1)
    assert torch.equal(got, want[:, 0])
    w.free()


@pytest.mark.parametrize("experts,top_k,hidden,inter,wtype,shared", [(16, 8, 768, 256, 12, False), (16, 4, 1280, 512, 13, True), (8, 8, 2816, 768, 12, False), (32, 8, 512, 256, 14, True)])
def test_few_experts_below_the_prefill_widths_match_eight_tokens_at_a_time(experts, top_k, hidden, inter, wtype, shared):
    """A dozen rows and more per expert take the GEMM from 17 tokens on: the layer and its two nodes against the same tokens handed
    over eight at a time, which never do."""
    import torch
    from densecore_amd import ops
    G, U = (ops.Q4KWeight.synthetic(s, inter, hidden, experts, wtype) for s in (1, 2))
    D = ops.Q4KWeight.synthetic(3, hidden, inter, experts, wtype)
    gen = torch.Generator(device="cuda").manual_seed(experts * top_k)
    sh = None
    if shared:
        sh = (ops.Q4KWeight.synthetic(4, inter, hidden, 1, wtype), ops.Q4KWeight.synthetic(5, inter, hidden, 1, wtype),
              ops.Q4KWeight.synthetic(6, hidden, inter, 1, wtype), torch.randn(hidden, device="cuda", generator=gen) * hidden ** -0.5)
    x, logits = torch.randn(191, hidden, device="cuda", generator=gen), torch.randn(191, experts, device="cuda", generator=gen)
    call = lambda a, b: ops.moe_layer(G, U, D, a, b, top_k, shared=sh, silu=ops.SILU_FAST)
    parts = [call(x[i:i + 8].contiguous(), logits[i:i + 8].contiguous()) for i in range(0, 191, 8)]
    want, want_ids, want_w = (torch.cat([p[j] for p in parts]) for j in range(3))
    hid = torch.cat([ops.moe_gateup_swiglu(G, U, x[i:i + 8].contiguous(), want_ids[i:i + 8].contiguous(), ops.SILU_FAST) for i in range(0, 191, 8)])
    for n in (24, 63, 96, 191):
        y, ids, w = call(x[:n].contiguous(), logits[:n].contiguous())
        assert torch.equal(ids, want_ids[:n]) and torch.equal(w, want_w[:n])
        # (a last-bit difference of a hidden value moves its 8-bit code by one now and then)
        assert ((y - want[:n]).norm() / want[:n].norm()).item() <= 2e-4, n
        h = ops.moe_gateup_swiglu(G, U, x[:n].contiguous(), ids, ops.SILU_FAST)
        assert (h - hid[:n]).abs().max().item() <= 1e-5 * hid.abs().max().item(), n
        d = ops.moe_down_weighted(D, hid[:n].contiguous(), ids, w)
        dw = torch.cat([ops.moe_down_weighted(D, hid[i:min(i + 8, n)].contiguous(), ids[i:min(i + 8, n)].contiguous(), w[i:min(i + 8, n)].contiguous()) for i in range(0, n, 8)])
        assert (d - dw).abs().max().item() <= 1e-5 * dw.abs().max().item(), n
    for t in (G, U, D) + (tuple(sh[:3]) if sh else ()):
        t.free()


def test_more_runs_of_rows_than_workgroups_quantize_them():
    """256 tiles of rows x 260 super-blocks are more than the launch has workgroups for: the second run of a workgroup, against halves that need none."""
    import torch
    from densecore_amd import ops
    experts, n, cols = 8, 4090, 260 * 256
    w = ops.Q4KWeight.synthetic(53, 16, cols, experts)
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn((n, cols), device="cuda", generator=gen)
    ids = torch.randint(0, experts, (n, 1), device="cuda", generator=gen, dtype=torch.int32)
    want = torch.cat([ops.mul_mat_id(w, x[i:i + 2045], ids[i:i + 2045]) for i in (0, 2045)])
    assert torch.equal(ops.mul_mat_id(w, x, ids), want)
    w.free()

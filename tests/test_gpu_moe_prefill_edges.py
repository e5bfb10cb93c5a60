"""Prefill-width forms of the kernels either side of the expert products, at the sizes where they change form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


def cu(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def into(ops, call, n, rows, shift):
    """y [n, rows] of call(pointer) written `shift` floats behind a 16-byte boundary."""
    import torch
    from densecore_amd import _lib
    buf = torch.full((n * rows + 8,), 7.0, device="cuda")
    _lib.check(call(buf.data_ptr() + 4 * shift), "call")
    assert bool((buf[:shift] == 7.0).all()) and bool((buf[shift + n * rows:] == 7.0).all())
    return buf[shift:shift + n * rows].view(n, rows).cpu().numpy()


@pytest.mark.parametrize("n,rows,k", [(512, 256, 3), (511, 256, 3), (256, 2048, 8), (300, 1280, 1), (520, 772, 2), (520, 770, 2)])
def test_combine_is_the_ordered_weighted_sum(ops, n, rows, k):
    """Four rows per thread from two workgroups per compute unit on; one row per thread below that, where rows % 4 != 0 and
    where y is not 16-byte aligned.  The products come from the same launch whatever the combine's form, and mul_mat_id gives
    the very rows the combine reads (both take the expert-grouped GEMM here), so every form equals the fp32 sum in routing
    order, formed on the host, to the last bit.  A slot of weight zero holds a row of infinities: it is skipped, not added."""
    import torch
    from densecore_amd import _lib
    experts = 8
    w = ops.Q4KWeight.synthetic(n * 7 + rows, rows, 256, experts)
    rng = np.random.default_rng(n + rows)
    ids = np.stack([rng.permutation(experts)[:k] for _ in range(n)]).astype(np.int32)
    wts = rng.random((n, k), dtype=np.float32)
    wts[3, 0] = 0.0              # skipped
    ids[5, k - 1] = experts + 2  # dropped
    hidden = torch.randn((n, k, 256), device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows))
    hidden[3, 0, 7] = float("inf")
    idd, wd = cu(ids), cu(wts)
    rows_out = ops.mul_mat_id(w, hidden, idd).cpu().numpy()
    want = np.zeros((n, rows), np.float32)
    for s in range(k):
        live = ((ids[:, s] >= 0) & (ids[:, s] < experts) & (wts[:, s] != 0))[:, None]
        with np.errstate(invalid="ignore"):
            want = np.where(live, want + rows_out[:, s] * wts[:, s:s + 1], want)
    assert np.isfinite(want).all()
    for shift in (0, 1, 4):
        got = into(ops, lambda y: _lib.lib().mq_moe_down_weighted_q4k(w._h, hidden.data_ptr(), n, idd.data_ptr(), wd.data_ptr(), k, y, ops._stream()),
                   n, rows, shift)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), shift
    w.free()


@pytest.mark.parametrize("n,hidden,gated", [(600, 512, True), (600, 512, False), (300, 1024, True)])
def test_combine_with_the_shared_expert(ops, n, hidden, gated):
    """The shared expert's row times its sigmoid gate joins behind the routed ones: four rows per thread (y aligned) and one row per
    thread (y not aligned) give the same bits, which are the routed part plus the gated FFN of the shared expert alone."""
    import ctypes as C

    import torch
    from densecore_amd import _lib
    inter, experts, k = 256, 8, 2
    G, U = (ops.Q4KWeight.synthetic(50 + i, inter, hidden, experts) for i in (1, 2))
    D = ops.Q4KWeight.synthetic(53, hidden, inter, experts)
    sg, su, sd = ops.Q4KWeight.synthetic(54, inter, hidden), ops.Q4KWeight.synthetic(55, inter, hidden), ops.Q4KWeight.synthetic(56, hidden, inter)
    gen = torch.Generator(device="cuda").manual_seed(n + hidden)
    x, lg = torch.randn((n, hidden), device="cuda", generator=gen), torch.randn((n, experts), device="cuda", generator=gen)
    gi = torch.randn(hidden, device="cuda", generator=gen) * hidden ** -0.5
    ids, wts = torch.empty((n, k), dtype=torch.int32, device="cuda"), torch.empty((n, k), device="cuda")
    d = _lib.MoELayerDesc(G._h, U._h, D._h, sg._h, su._h, sd._h, gi.data_ptr() if gated else None, k, ops.SILU_FAST, ops.ROUTE_FUSED)
    got = [into(ops, lambda y: _lib.lib().mq_moe_layer_q4k(C.byref(d), x.data_ptr(), lg.data_ptr(), n, y, ids.data_ptr(), wts.data_ptr(), ops._stream()),
                n, hidden, shift) for shift in (0, 1)]
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    routed = ops.moe_layer(G, U, D, x, lg, k, silu=ops.SILU_FAST)[0].double()
    alone = ops.ffn_swiglu(sg, su, sd, x, ops.SILU_FAST_FMA).double()
    gate = torch.sigmoid(x.double() @ gi.double())[:, None] if gated else 1.0
    want = (routed + gate * alone).cpu().numpy()
    # the FFN entry's kernels sum a product in another order, which now and then moves an 8-bit code of a hidden row by one: at most
    # 1 / 254 of the row's largest value on one of its 256, so 4e-3 of the outputs' scale and far less on average
    scale = np.abs(want).max()
    assert np.abs(got[0] - want).max() <= 4e-3 * scale and np.sqrt(np.mean((got[0] - want) ** 2)) <= 2e-4 * np.sqrt(np.mean(want ** 2))
    for w in (G, U, D, sg, su, sd):
        w.free()


def grouped(ops, ids, experts):
    from oracle import binding as orc
    assert np.array_equal(ops.debug_moe_groups(experts, ids.shape[1], ids=cu(ids)), orc.build_assignments(ids, experts))


@pytest.mark.parametrize("n,experts,k", [(1, 4, 2), (31, 7, 3), (32, 4, 4), (33, 250, 8), (96, 300, 8), (127, 8, 8), (129, 8, 8), (545, 16, 5), (2047, 255, 8),
                                         (4096, 5, 3), (1500, 1100, 8)])
def test_group_lists_from_masks(ops, n, experts, k):
    """One to 128 mask words, divided over four lanes with and without a remainder; experts not a multiple of the lanes'; pairs up to and
    past the eight rounds requested together; masks that leave no room (1100 experts): the lists are whole numbers, so equal."""
    rng = np.random.default_rng(n + experts)
    grouped(ops, np.stack([rng.permutation(experts)[:k] for _ in range(n)]).astype(np.int32), experts)


@pytest.mark.parametrize("n,experts,k", [(33, 9, 4), (150, 9, 8), (1200, 64, 8)])
def test_group_lists_with_one_repeat_in_the_last_token(ops, n, experts, k):
    """A single repeated (token, expert) sends the whole list to the scan, with dropped ids on the way."""
    rng = np.random.default_rng(n)
    ids = np.stack([rng.permutation(experts)[:k] for _ in range(n)]).astype(np.int32)
    ids[n - 1, k - 1] = ids[n - 1, 0]
    ids[n // 2, 0], ids[0, k - 1] = -1, experts
    grouped(ops, ids, experts)


@pytest.mark.parametrize("n", [191, 192, 193])
def test_route_then_group_from_1536_pairs(ops, n):
    """The change from one launch that routes and groups to two, at 8 experts of 256 per token."""
    from densecore_amd import synth
    from oracle import binding as orc
    logits = synth.normal_f32(synth.tensor_seed("edge", n), (n, 256))
    ids, _ = orc.route_topk(logits, 8, 0)
    assert np.array_equal(ops.debug_moe_groups(256, 8, logits=cu(logits)), orc.build_assignments(ids, 256))

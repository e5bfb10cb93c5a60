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


@pytest.mark.parametrize("n,rows,k", [(512, 256, 3), (511, 256, 3), (256, 2048, 8), (300, 1280, 1), (520, 772, 2), (520, 770, 2)])
def test_combine_is_the_ordered_weighted_sum(ops, n, rows, k):
    """Four rows per thread from two workgroups per compute unit on (one row per
    thread below that and where rows % 4 != 0).  The products themselves come from mul_mat_id, so only the combine differs: k fp32 products and sums in
    routing order, formed here in float32 the same way, equal to the last bit where both run on the same kernel and within
    the order of one fp32 sum over 256 weights (2^-23 * 16 partial sums, of values of order one) where they do not."""
    import torch
    experts = 8
    w = ops.Q4KWeight.synthetic(n * 7 + rows, rows, 256, experts)
    rng = np.random.default_rng(n + rows)
    ids = np.stack([rng.permutation(experts)[:k] for _ in range(n)]).astype(np.int32)
    wts = rng.random((n, k), dtype=np.float32)
    wts[3, 0] = 0.0              # skipped
    ids[5, k - 1] = experts + 2  # dropped
    hidden = torch.randn((n, k, 256), device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows))
    got = ops.moe_down_weighted(w, hidden, cu(ids), cu(wts)).cpu().numpy()
    rows_out = ops.mul_mat_id(w, hidden, cu(ids)).cpu().numpy()
    want = np.zeros((n, rows), np.float32)
    for s in range(k):
        live = ((ids[:, s] >= 0) & (ids[:, s] < experts) & (wts[:, s] != 0))[:, None]
        want = np.where(live, want + rows_out[:, s] * wts[:, s:s + 1], want)
    scale = np.sqrt(np.mean(want ** 2)) + 1e-30
    assert np.max(np.abs(got - want)) <= 16 * 2.0 ** -23 * max(8.0, np.max(np.abs(want)) / scale) * scale


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

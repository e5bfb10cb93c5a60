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

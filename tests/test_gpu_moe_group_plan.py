"""Grouping and plan of the expert-grouped GEMM in one launch (a workgroup per expert) and, beyond its limits, in two: every
(token, slot) row of mul_mat_id must be the product of its own expert, whatever the ids hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch
    from densecore_amd import ops as o
    assert torch.cuda.is_available()
    return o


# experts: one, few, not a multiple of a wavefront's lanes, the last count that takes the one launch and the first that does not;
# pairs: a last run of ids of one pair, 64 runs of 1024 pairs in full and one token more
@pytest.mark.parametrize("n,experts,k,per_slot", [(193, 1, 1, False), (205, 5, 5, True), (400, 7, 3, False), (192, 256, 8, True), (700, 300, 8, False),
                                                  (400, 512, 8, False), (400, 513, 8, False), (8192, 4, 8, False), (8193, 4, 8, False)])
def test_every_row_is_its_own_experts_product(ops, n, experts, k, per_slot):
    """The rows of an expert multiplied by themselves (a stack of one expert, the same kernel and order of sums) are the reference: equal
    to the bit.  Ids are repeated within a token, dropped (negative, one past the last expert), and one expert gets none."""
    import torch
    from densecore_amd import synth
    rows, cols = 64, 256
    blocks = np.stack([synth.q4k_matrix(n + e, rows, cols) for e in range(experts)])
    rng = np.random.default_rng(n + experts)
    ids = rng.integers(0, experts, (n, k)).astype(np.int32)
    if experts > 2:
        ids[ids == experts // 2] = 0  # a group that is empty
    ids[3, 0], ids[n // 2, k - 1], ids[n - 1, 0] = -1, experts, experts - 1
    x = torch.randn((n, k, cols) if per_slot else (n, cols), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    w = ops.Q4KWeight.from_ggml(blocks, cols)
    idd = torch.from_numpy(ids).cuda()
    y = ops.mul_mat_id(w, x, idd)
    live = (idd >= 0) & (idd < experts)
    assert bool((y[~live] == 0).all())
    for e in sorted({0, experts - 1, experts // 3, experts // 2}):
        tok, slot = torch.nonzero(idd == e, as_tuple=True)
        if len(tok) == 0:
            continue
        one = ops.Q4KWeight.from_ggml(blocks[e:e + 1], cols)
        xe = x[tok, slot] if per_slot else x[tok]
        xe = torch.cat([xe, xe.new_zeros((max(0, 192 - len(tok)), cols))])  # wide enough for the grouped GEMM
        want = ops.mul_mat_id(one, xe, torch.zeros((len(xe), 1), dtype=torch.int32, device="cuda"))[:len(tok), 0]
        assert torch.equal(y[tok, slot], want), e
        one.free()
    w.free()

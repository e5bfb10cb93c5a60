"""GPU: Q8_0 GEMM with K in runs (few workgroups, long rows), and the tiles to a workgroup of a matrix of many rows at few activation rows."""
import pytest

from densecore_amd import synth
from tests._parity import GEMM, dense_path, gemm_launch, gemm_shape

pytestmark = pytest.mark.gpu
Q80 = synth.GGML_TYPE_Q8_0


# row counts that leave 0 .. 3 rows beside whole groups of four, an odd last run, up to sixteen runs; one and two tiles to a workgroup
@pytest.mark.parametrize("rows,cols,n,tiles,runs", [(64, 16384, 100, 1, 16), (65, 16384, 40, 1, 16), (527, 12544, 148, 1, 5), (529, 8192, 33, 1, 8), (1866, 10240, 27, 1, 8),
                                                    (1003, 2048, 40, 1, 1), (6315, 6912, 15, 1, 5), (33001, 256, 10, 1, 1), (65536, 512, 17, 2, 1), (66000, 256, 31, 2, 1)])
def test_matches_eight_rows_at_a_time(rows, cols, n, tiles, runs):
    """Block sums are integers in both; the scaled blocks are added up in fp32 in another order: 2 K / 32 roundings of 2^-24 of the largest result
    at most.  A captured launch gives the eager one's bits at each replay."""
    import torch
    from densecore_amd import _lib, ops
    path, _, mt = dense_path(Q80, rows, cols // 256, n)
    assert (path, mt) == (GEMM, tiles) and gemm_launch(Q80, rows, cols, n)["runs"] == runs
    w = ops.Q4KWeight.synthetic(rows + n, rows, cols, 1, Q80)
    x = torch.randn(n, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    want = torch.cat([ops.mul_mat(w, x[i:i + 8]) for i in range(0, n, 8)])
    wide = torch.full((n + 1, rows + 3), 7.0, device="cuda")
    _lib.check(_lib.lib().mq_mul_mat_q4k(w._h, x.data_ptr(), n, cols, wide.data_ptr(), rows + 3, torch.cuda.current_stream().cuda_stream), "mq_mul_mat_q4k")
    got = wide[:n, :rows]
    assert (got - want).abs().max().item() <= 2 * cols / 32 * 2.0 ** -24 * want.abs().max().item()
    assert bool((wide[:n, rows:] == 7.0).all()) and bool((wide[n] == 7.0).all())
    side, out, graph = torch.cuda.Stream(), torch.empty(n, rows, device="cuda"), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.mul_mat(w, x, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)
    w.free()


@pytest.mark.parametrize("wtype,rows", [(Q80, 2000), (12, 2001), (12, 2000)])
def test_planes_that_cannot_grow_under_capture_leave_k_whole(wtype, rows):
    """No eager call had this matrix (one of four rows made room for the activations alone): the captured product, whose runs would need
    planes, is taken all the same, with K whole, and its sums are in another order than the eager one's."""
    import torch
    from densecore_amd import _lib, ops
    torch.cuda.synchronize()
    _lib.check(_lib.lib().mq_shutdown(), "mq_shutdown")  # gives the workspaces back
    _lib.check(_lib.lib().mq_init(torch.cuda.current_device()), "mq_init")
    cols, n, padded = 16384, 100, (rows + 3) // 4 * 4
    assert wtype == Q80 or gemm_shape(wtype, padded, cols, 4096)["runs"] == 1
    assert gemm_launch(wtype, rows, cols, n)["runs"] > 1
    w, other = (ops.Q4KWeight.synthetic(rows, r, cols, 1, wtype) for r in (rows, 4))
    x = torch.randn(4096, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    ops.mul_mat(other, x)
    side, out, graph = torch.cuda.Stream(), torch.empty(n, rows, device="cuda"), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.mul_mat(w, x[:n], out)
    graph.replay()
    want = ops.mul_mat(w, x[:n])
    torch.cuda.synchronize()
    assert (out - want).abs().max().item() <= 2 * cols / 32 * 2.0 ** -24 * want.abs().max().item()
    assert not torch.equal(out, want)
    for m in (w, other):
        m.free()

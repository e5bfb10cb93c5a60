"""mq_mul_mat_q4k_noalloc, the entry point for callers that cannot allocate: called through the C ABI, its outputs
must equal mq_mul_mat_q4k's bit for bit -- on two calls in a row, the second with a smaller input (the fixed scratch
keeps the first call's contents), for each weight type, and sizes beyond the scratch must be refused."""
import numpy as np
import pytest

from densecore_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from densecore_amd import _lib, ops
    assert torch.cuda.is_available()
    return torch, _lib, ops


def _both(env, W, x):
    """(existing entry point, allocation-free entry point) outputs for the rows x."""
    torch, _lib, ops = env
    n = x.shape[0]
    want = ops.mul_mat(W, x)
    got = torch.full((n, W.rows), float("nan"), dtype=torch.float32, device=x.device)
    rc = _lib.lib().mq_mul_mat_q4k_noalloc(W._h, x.data_ptr(), n, x.stride(0), got.data_ptr(), W.rows, None)
    _lib.check(rc, "mq_mul_mat_q4k_noalloc")
    torch.cuda.synchronize()
    return want.cpu().numpy(), got.cpu().numpy()


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,n_first,n_second", [(2048, 2048, 16, 3), (4096, 4096, 8, 1), (14336, 4096, 5, 2),
                                                        (100, 16384, 16, 9), (4096, 14336, 1, 1)])
def test_two_calls_in_a_row_equal_the_allocating_entry_point(env, wtype, rows, cols, n_first, n_second):
    torch, _lib, ops = env
    W = ops.Q4KWeight.synthetic(synth.tensor_seed("noalloc", wtype, rows, cols), rows, cols, ggml_type=wtype)
    for n in (n_first, n_second):
        x = torch.from_numpy(synth.normal_f32(synth.tensor_seed("noalloc-x", rows, cols, n), (n, cols))).cuda()
        want, got = _both(env, W, x)
        assert np.array_equal(want.view(np.uint32), got.view(np.uint32)), f"n={n}: outputs differ"


@pytest.mark.parametrize("wtype", [12, 13, 14])
@pytest.mark.parametrize("rows,cols", [(5120, 11008), (14336, 11008), (8704, 9472), (2048, 5632)])
def test_rows_of_uneven_super_blocks_equal_the_allocating_entry_point(env, wtype, rows, cols):
    """Long rows that no useful wavefront count divides, where other kernels take a product from nine or seventeen rows on."""
    torch, _lib, ops = env
    W = ops.Q4KWeight.synthetic(synth.tensor_seed("noalloc-u", wtype, rows, cols), rows, cols, ggml_type=wtype)
    x = torch.from_numpy(synth.normal_f32(synth.tensor_seed("noalloc-ux", rows, cols), (16, cols))).cuda()
    for n in (8, 9, 16):
        want, got = _both(env, W, x[:n])
        assert np.array_equal(want.view(np.uint32), got.view(np.uint32)), f"n={n}: outputs differ"
    W.free()


def test_smaller_matrix_after_larger_one(env):
    """A 16384-column product fills the whole scratch; a 256-column one after it reads only its own corner."""
    torch, _lib, ops = env
    big = ops.Q4KWeight.synthetic(11, 64, 16384)
    small = ops.Q4KWeight.synthetic(12, 48, 256)
    for W, n in ((big, 16), (small, 2), (big, 1)):
        x = torch.from_numpy(synth.normal_f32(synth.tensor_seed("noalloc-y", W.cols, n), (n, W.cols))).cuda()
        want, got = _both(env, W, x)
        assert np.array_equal(want.view(np.uint32), got.view(np.uint32))


def test_sizes_beyond_the_scratch_are_refused(env):
    torch, _lib, ops = env
    W = ops.Q4KWeight.synthetic(13, 32, 512)
    x = torch.zeros((17, 512), dtype=torch.float32, device="cuda")
    y = torch.zeros((17, 32), dtype=torch.float32, device="cuda")
    rc = _lib.lib().mq_mul_mat_q4k_noalloc(W._h, x.data_ptr(), 17, 512, y.data_ptr(), 32, None)
    assert rc != 0 and b"exceed" in _lib.lib().mq_last_error()
    wide = ops.Q4KWeight.synthetic(14, 16, 16384 + 256)
    xw = torch.zeros((1, 16384 + 256), dtype=torch.float32, device="cuda")
    rc = _lib.lib().mq_mul_mat_q4k_noalloc(wide._h, xw.data_ptr(), 1, 16384 + 256, y.data_ptr(), 32, None)
    assert rc != 0 and b"exceed" in _lib.lib().mq_last_error()
    rc = _lib.lib().mq_mul_mat_q4k_noalloc(W._h, x.data_ptr(), 0, 512, y.data_ptr(), 32, None)
    assert rc == 0  # an empty product is fine

"""GPU tests of row_sum_kernel (NnClGlob.Sum over the last axis): one launch or chunk sums,
rows ending inside a tile of 64 columns or a chunk of 256, rows off 16-byte boundaries. The
bits must be those of the documented order: 256 values at a time ascending from +0.0f, the
chunk sums added in chunk order."""
import ctypes

import numpy as np
import pytest
import torch

from my_pytchon_opencl_lib_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,axis", [(64, 16), (65, 63), (130, 64), (200, 255), (64, 256),
                                       (77, 257), (129, 1024), (100, 1025), (70, 5000),
                                       (32769, 1283)])
def test_row_sums_bit_for_bit(nncl, rows, axis):
    print("row sum", rows, axis, flush=True)
    rng = np.random.default_rng(rows + axis)
    x = rng.standard_normal((rows, axis)).astype(np.float32)
    x[0, 0], x[1, axis - 1], x[2, 3] = np.inf, np.nan, -0.0
    expect = None
    for a in range(0, axis, 256):
        s = np.cumsum(x[:, a:a + 256], axis=1, dtype=np.float32)[:, -1]
        expect = s if expect is None else expect + s
    buf = torch.full((rows * axis + 1,), float("nan"), device="cuda:0")
    for off in (0, 1):  # the second time every row starts 4 bytes off
        t = buf[off:off + rows * axis].view(rows, axis)
        t.copy_(torch.from_numpy(x))
        got = nncl.Sum(t, 1).cpu().numpy()
        assert _native.last_plan().startswith("row_sum"), _native.last_plan()
        assert np.array_equal(got, expect, equal_nan=True)


def test_short_or_few_rows_keep_the_column_kernel(nncl):
    for rows, axis in [(63, 400), (500, 15)]:
        t = torch.ones(rows, axis, device="cuda:0")
        assert torch.equal(nncl.Sum(t, 1), torch.full((rows,), float(axis), device="cuda:0"))
        assert _native.last_plan().startswith("column_sum"), _native.last_plan()


@pytest.mark.parametrize("rows,kernel", [((1 << 30) - 64, "row_sum"), (1 << 30, "column_sum")])
def test_more_rows_than_one_launch_holds(nncl, rows, kernel):
    """row_sum_kernel starts 4 threads per row: 2^30 rows need 2^32, one more than a grid
    holds, and run through the column kernel (64 GiB of values)."""
    print("rows of one launch", rows, flush=True)
    t = torch.empty(rows, 16, device="cuda:0")
    t.copy_(torch.arange(16.0, device="cuda:0"))
    t[rows - 1] = 2.0
    got = nncl.Sum(t, 1)
    assert _native.last_plan().startswith(kernel + " "), _native.last_plan()
    assert float(got[rows - 1]) == 32.0
    assert bool((got[:rows - 1] == 120.0).all())
    del t, got
    torch.cuda.empty_cache()


def test_whole_rows_are_captured_without_a_workspace(nncl):
    """A work-group that sums whole rows keeps no chunk sums: captured on a stream that holds
    no workspace, replays agree with the eager sum."""
    t = torch.randn(32768, 1283, device="cuda:0")
    expect = nncl.Sum(t, 1)
    cap = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        got = nncl.Sum(t, 1)
    for _ in range(3):
        got.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, expect)
    size = ctypes.c_size_t(1)
    _native.call("migemm_workspace_size", ctypes.c_void_p(cap.cuda_stream), ctypes.byref(size))
    assert size.value == 0

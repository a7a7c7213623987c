"""Recorded launches: up to five go out one by one, more as a graph, and so does what is no chain of kernels."""
import ctypes

import numpy as np
import pytest

from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('memcpy_at', [None, 0, 2])
@pytest.mark.parametrize('n', [1, 2, 64, 65])
def test_replays_run_every_launch_in_order(n, memcpy_at):
    """A value handed from buffer to buffer by n launches arrives in the last one, at every replay."""
    hk.init(0)
    L = hk.lib()
    bufs = [hk.DeviceBuffer.from_numpy(np.full(256, -i, np.int32)) for i in range(n + 1)]
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    hk.check(L.pml_hip_stream_create(ctypes.byref(stream)))
    hk.check(L.pml_hip_capture_begin(stream))
    for i in range(n):
        if i == memcpy_at:
            hk.check(L.pml_hip_memcpy_d2d(bufs[i + 1].ptr, bufs[i].ptr, 1024, stream))
        else:
            dst, src, size = hk.ptr_array([bufs[i + 1].ptr]), hk.ptr_array([bufs[i].ptr]), (ctypes.c_size_t * 1)(1024)
            hk.check(L.pml_hip_copy_spans(1, dst, src, size, stream))
    hk.check(L.pml_hip_capture_end(stream, ctypes.byref(graph)))
    try:
        np.testing.assert_array_equal(bufs[n].to_numpy(np.int32, (256,)), -n)  # (recorded, not run)
        for turn in range(4):
            x = np.arange(256, dtype=np.int32) * (turn + 3)
            hk.check(L.pml_hip_memcpy_h2d(bufs[0].ptr, x.ctypes.data_as(ctypes.c_void_p), 1024, stream))
            hk.check(L.pml_hip_graph_launch(graph, stream))
            hk.check(L.pml_hip_stream_sync(stream))
            np.testing.assert_array_equal(bufs[n].to_numpy(np.int32, (256,)), x)
    finally:
        hk.check(L.pml_hip_graph_destroy(graph))
        hk.check(L.pml_hip_stream_destroy(stream))


@pytest.mark.parametrize('memcpy_at', [None, 0, 2])
@pytest.mark.parametrize('n', [5, 6])
def test_replays_on_both_sides_of_one_by_one(n, memcpy_at):
    test_replays_run_every_launch_in_order(n, memcpy_at)

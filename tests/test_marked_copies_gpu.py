"""Copies by kernel that leave a mark in host memory: the host that sees the mark sees what was copied."""
import ctypes

import numpy as np
import pytest

from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


# no copy, one, a full launch, a launch and one, three launches; bytes of less than a vector up to 64 workgroups a copy
@pytest.mark.parametrize('n', [0, 1, 16, 17, 40])
@pytest.mark.parametrize('nbytes', [3, 16384, 300001])
def test_what_is_marked_is_there(n, nbytes):
    hk.init(0)
    L = hk.lib()
    host, arrived = ctypes.c_void_p(), hk.DeviceBuffer.from_numpy(np.zeros(1, np.uint32))
    pitch = (nbytes + 255) // 256 * 256
    hk.check(L.pml_hip_host_alloc(ctypes.byref(host), 256 + pitch * max(1, n)))
    mark = ctypes.cast(host, ctypes.POINTER(ctypes.c_uint32))
    mark[0] = 0
    landed = np.ctypeslib.as_array(ctypes.cast(host, ctypes.POINTER(ctypes.c_uint8)), (256 + pitch * max(1, n),))[256:].reshape(-1, pitch)
    stream = ctypes.c_void_p()
    hk.check(L.pml_hip_stream_create(ctypes.byref(stream)))
    try:
        for turn in range(1, 21):
            x = np.random.default_rng(turn).integers(0, 255, (max(1, n), pitch), dtype=np.uint8)
            dev = hk.DeviceBuffer.from_numpy(x)
            dst = hk.ptr_array([host.value + 256 + i * pitch for i in range(n)], 64)
            src = hk.ptr_array([dev.ptr + i * pitch for i in range(n)], 64)
            sizes = (ctypes.c_size_t * max(1, n))(*[nbytes] * n)
            hk.check(L.pml_hip_copy_spans_marked(n, dst, src, sizes, None, mark, arrived.ptr, turn, stream))
            hk.check(L.pml_hip_wait_mark(mark, turn, stream))
            got = landed[:n, :nbytes].copy()
            assert mark[0] == turn
            np.testing.assert_array_equal(got, x[:n, :nbytes])
            hk.check(L.pml_hip_stream_sync(stream))
        hk.check(L.pml_hip_wait_mark(mark, 99, stream))  # a mark that nobody leaves: the end of the stream
    finally:
        hk.check(L.pml_hip_stream_sync(stream))
        hk.check(L.pml_hip_stream_destroy(stream))
        L.pml_hip_host_free(host)

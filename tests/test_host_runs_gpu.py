"""Runs on arrays in host memory (host/src/hip_runtime.cc, Runner) around the edges of their staging."""
import ctypes

import numpy as np
import pytest

from plaidml_amd import edsl as P
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
DT = {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16}


def test_an_allocation_that_fails_does_not_fail_the_next_launch():
    L = hk.lib()
    hk.init(0)
    ptr = ctypes.c_void_p()
    assert L.pml_hip_malloc(ctypes.byref(ptr), 1 << 50) != 0 and b'hipMalloc' in L.pml_hip_last_error()
    buf = hk.DeviceBuffer(4096)
    hk.check(L.pml_hip_fill_u32(buf.ptr, 0x01020304, 1024, None))
    np.testing.assert_array_equal(buf.to_numpy(np.uint32, (1024,)), 0x01020304)

"""What a plan's text says about the kernel that runs.  Plans over [N][K] right-hand sides hold no memory: no device needed."""
import ctypes

import pytest

from plaidml_amd import hipkernels as hk


def text(m, n, k, dt=hk.BF16, lda=None, ldr=None, flags=0, c=None):
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = dt, c or (hk.I32 if dt == hk.I8 else dt), c or (hk.I32 if dt == hk.I8 else dt)
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = m, n, k, lda or k, k, n, 1, flags
    if ldr is not None:
        d.tail = hk.make_tail(ops=[(hk.EPI_ADD, dt, hk.OPND_TENSOR, 0, 0.0)], operands=[(dt, ldr, 1)])
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, hk.lib().pml_hip_last_error()
    try:
        return hk.describe(plan)
    finally:
        hk.lib().pml_hip_plan_free(plan)


def test_streamed_rows_are_named():
    assert text(401408, 256, 64).endswith(', streamed rows past B mfma=f32_16x16x32_bf16')
    # a named tile is taken; so is one for other types, for long rows, for residual rows off eight bytes
    for other in (text(401408, 256, 64, flags=hk.flag_tile('128x128w8s2')), text(401408, 256, 64, c=hk.F32), text(401408, 256, 264), text(401408, 256, 64, dt=hk.I8),
                  text(401408, 256, 64, ldr=257)):
        assert 'streamed' not in other, other
    assert 'streamed' in text(401408, 255, 64, ldr=256)


@pytest.mark.parametrize('dt,mfma', [(hk.F32, 'f32_16x16x4'), (hk.BF16, 'f32_16x16x32_bf16'), (hk.I8, 'i32_16x16x64_i8')])
def test_direct_tiles_name_their_instruction(dt, mfma):
    assert text(49, 512, 512, dt=dt).endswith('(8 wavefronts sharing K) mfma=' + mfma)


# (both sides of each line of the rule, products that were timed on both sides of it; a device of 256 compute units, which is
# also what is assumed where there is none)
@pytest.mark.parametrize('m,n,k,lda,ldr,takes', [
    (24576, 256, 32, 32, None, True), (24560, 256, 32, 32, None, False), (25088, 256, 64, 64, None, False), (69632, 256, 64, 64, None, True), (69616, 256, 64, 64, None, False),
    (25088, 512, 128, 128, None, False), (100352, 64, 128, 128, None, False), (100352, 512, 128, 128, None, True), (25088, 256, 200, 200, None, False),
    (25088, 256, 200, 200, 256, True), (100352, 64, 200, 200, None, True), (100352, 64, 200, 256, None, False), (26624, 256, 200, 200, None, True),
    (26608, 256, 200, 200, None, False), (25088, 251, 200, 200, None, True), (12544, 1024, 256, 256, None, False), (25088, 1024, 256, 256, None, True),
    (25088, 512, 256, 256, 512, True), (25088, 512, 256, 256, None, False), (35000, 250, 256, 256, None, True), (25088, 512, 256, 264, None, True)])
def test_which_rows_stream(m, n, k, lda, ldr, takes):
    got = text(m, n, k, lda=lda, ldr=ldr)
    assert ('streamed' in got) == takes, got

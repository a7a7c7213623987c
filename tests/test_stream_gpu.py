"""bf16 products whose rows stream past a right-hand side in registers (csrc/stream.hip).  Small whole numbers make every sum
exact, so every tail is compared value for value with numpy, where rows, columns and K end raggedly."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _device():
    hk.init(0)


def whole(rng, shape):
    return rng.integers(-4, 5, shape).astype(np.float32)


# rows: one past and one short of a step, more than one round of the device; columns: fewer than a wavefront holds, that end
# within a quarter, a pair, a wavefront, a workgroup; K: one chunk, just below, at and above each kernel's range
@pytest.mark.parametrize('M,N,K', [(80000, 72, 8), (73000, 256, 64), (70001, 200, 72), (34832, 512, 128), (36399, 264, 136), (320001, 40, 256), (140000, 8, 248), (17000, 1160, 56)])
def test_tails(M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    S = A @ B  # at most 16 K: exact
    bias, res = whole(rng, N), whole(rng, (M, N))
    A[M - 1, K - 1] = A[0, 0] = np.inf  # (in its own row only)
    with np.errstate(invalid='ignore'):
        S[[0, M - 1]] = A[[0, M - 1]] @ B
    r = E.round_bf16
    relu = (hk.EPI_RELU, hk.BF16, 0, 0, 0.0)
    bits = (T.bf16(A), T.bf16(B), hk.BF16, hk.BF16)
    kw = dict(init=T.bf16(bias), init_strides=(0, 1), init_dt=hk.BF16, invokes=2)

    def check(got, want):
        np.testing.assert_array_equal(E.bf16_from_bits(got), want)
    check(T.run_gemm(*bits), r(S))
    with np.errstate(invalid='ignore'):
        keep = lambda v: np.where(v < 0, np.float32(0), v)  # (relu keeps a NaN)
        check(T.run_gemm(*bits, tail=hk.make_tail(ops=[relu]), **kw), r(keep(S + bias)))
        add = hk.make_tail(ops=[(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0), relu], operands=[(hk.BF16, N, 1)])
        check(T.run_gemm(*bits, tail=add, operands=[T.bf16(res)], **kw), r(keep(r(S + bias) + res)))


@pytest.mark.parametrize('stride', [0, 1])
@pytest.mark.parametrize('M,N,K,K2', [(81920, 256, 64, 64), (143360, 72, 32, 96), (73728, 136, 96, 24)])
def test_second_product(M, N, K, K2, stride):
    rng = np.random.default_rng(M + K2)
    A, B, A2, B2 = whole(rng, (M, K)), whole(rng, (K, N)), whole(rng, (M, K2)), whole(rng, (K2, N))
    b1, b2 = whole(rng, N), whole(rng, N)
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = d.init_dtype = hk.BF16
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.k2, d.lda2, d.ldb2 = M, N, K, K, N, N, K2, K2, N
    d.init_kind = d.init_col_stride = d.init2_kind = 1
    if stride:
        d.a2_stride, d.a2_h, d.a2_w, d.a2_oh, d.a2_ow = 1, 64, 64, 64, 64
    d.tail = hk.make_tail(ops=[(hk.EPI_RELU, hk.BF16, 0, 0, 0.0)])
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan
    dA, dB, dA2, dB2, d1, d2 = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, B, A2, B2, b1, b2))
    dC, none = hk.DeviceBuffer(M * N * 2), hk.ptr_array([])
    hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr, None))
    hk.check(L.pml_hip_gemm_pack_b2(plan, dB2.ptr, None))
    hk.check(L.pml_hip_gemm_invoke2(plan, dA.ptr, None, dC.ptr, d1.ptr, dA2.ptr, None, d2.ptr, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (M, N))), E.round_bf16(np.maximum(A @ B + A2 @ B2 + b1 + b2, 0)))
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('n,hw,ci,co', [(45, 56, 64, 72), (33, 40, 128, 264), (40, 61, 200, 64)])
def test_one_by_one_convolution(n, hw, ci, co):
    rng = np.random.default_rng(ci + co)
    X, F, bias = whole(rng, (n, hw, hw, ci)), whole(rng, (1, 1, ci, co)), whole(rng, co)
    d = hk.Conv2dDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = d.init_dtype = hk.BF16
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, hw, hw, ci, 1, 1, co, hw, hw
    d.stride_h = d.stride_w = d.dil_h = d.dil_w = d.init_kind = d.init_col_stride = 1
    L = hk.lib()
    plan = L.pml_hip_conv2d_dispatch(ctypes.byref(d))
    assert plan
    dX, dF, d1 = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (X, F, bias))
    dC, none = hk.DeviceBuffer(n * hw * hw * co * 2), hk.ptr_array([])
    hk.check(L.pml_hip_conv2d_invoke(plan, dX.ptr, dF.ptr, dC.ptr, d1.ptr, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    want = E.round_bf16(X.reshape(-1, ci) @ F.reshape(ci, co) + bias)
    np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (n * hw * hw, co))), want)
    L.pml_hip_plan_free(plan)

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


def spread(x, pitch, at=0):
    """Rows `pitch` values apart from the `at`-th value on, NaNs between them."""
    flat = np.full(at + x.shape[0] * pitch, np.nan, np.float32)
    flat[at:].reshape(-1, pitch)[:, :x.shape[1]] = x
    return flat


def run(A, B, packed, at=0, pitch=None, bias=None, res=None, relu=False, lda=0, ldb=0, ldr=0, b_at=0):
    """Result rows `pitch` values apart that begin `at` values behind a 16-byte boundary, and whether all else was left alone.
    Rows of the operands lie whole behind one another, or `lda`, `ldb`, `ldr` values apart; those of the residual tensor on
    8-byte boundaries (any others take a tile and the interpreted tail).  B begins `b_at` values behind a boundary.  The plan's
    text has to name the kernel."""
    (M, K), N = A.shape, B.shape[1]
    pitch, lda, ldb, ldr = pitch or N, lda or K, ldb or N, ldr or (N + 3) // 4 * 4
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = d.init_dtype = hk.BF16
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.init_kind, d.init_col_stride = M, N, K, lda, ldb, pitch, int(bias is not None), 1
    ops = [(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0)] * (res is not None) + [(hk.EPI_RELU, hk.BF16, 0, 0, 0.0)] * relu
    d.tail = hk.make_tail(ops=ops, operands=[(hk.BF16, ldr, 1)] * (res is not None))
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan
    text = hk.describe(plan)
    assert ('streamed rows past B packed' if packed or K > 128 else 'as it lies mfma') in text and 'streamed' in text, text
    dA, dB = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (spread(A, lda), spread(B, ldb, b_at)))
    d1, dR = (hk.DeviceBuffer.from_numpy(T.bf16(x)) if x is not None else None for x in (bias, None if res is None else spread(res, ldr)))
    n = (at + M * pitch + 9) // 2 * 2
    dC = hk.DeviceBuffer(n * 2)
    hk.check(L.pml_hip_fill_u32(dC.ptr, 0xbeefbeef, n // 2, None))
    if packed:
        hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr + 2 * b_at, None))
    for _ in range(2):
        hk.check(L.pml_hip_gemm_invoke(plan, dA.ptr, None if packed else dB.ptr + 2 * b_at, dC.ptr + 2 * at, d1.ptr if d1 else None, hk.ptr_array([dR.ptr] if dR else []),
                                       hk.ptr_array([]), None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(plan)
    flat = dC.to_numpy(np.uint16, (n,))
    rows = flat[at:at + M * pitch].reshape(M, pitch)
    assert (flat[:at] == 0xbeef).all() and (flat[at + M * pitch:] == 0xbeef).all() and (rows[:, N:] == 0xbeef).all()
    return E.bf16_from_bits(np.ascontiguousarray(rows[:, :N]))


# rows: one past and one short of a step, more than one round of the device; columns: fewer than a wavefront holds, that end
# within eight, a quarter, a pair, a wavefront, a workgroup; K: one chunk, just below, at and above each kernel's range; result
# rows with and without room behind them that begin on 16 bytes, a word, half a word
@pytest.mark.parametrize('packed', [0, 1])
@pytest.mark.parametrize('M,N,K,at,pitch', [
    (80000, 72, 8, 0, 72), (73000, 256, 64, 0, 256), (70001, 200, 72, 0, 208), (34832, 512, 128, 0, 512), (36399, 264, 136, 0, 264), (320001, 40, 256, 0, 40),
    (17000, 1160, 56, 0, 1160), (80000, 76, 24, 0, 76), (140000, 1, 64, 1, 1), (73000, 260, 40, 2, 263), (140001, 7, 96, 0, 9), (69999, 132, 128, 1, 132),
    (36399, 250, 248, 3, 250), (320001, 60, 256, 0, 60)])
def test_tails(M, N, K, at, pitch, packed):
    rng = np.random.default_rng(M + N + K)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    S = A @ B  # at most 16 K: exact
    bias, res = whole(rng, N), whole(rng, (M, N))
    A[M - 1, K - 1] = A[0, 0] = np.inf  # (in its own row only)
    r = E.round_bf16
    with np.errstate(invalid='ignore'):
        S[[0, M - 1]] = A[[0, M - 1]] @ B
        keep = lambda v: np.where(v < 0, np.float32(0), v)  # (relu keeps a NaN)
        np.testing.assert_array_equal(run(A, B, packed, at, pitch), r(S))
        np.testing.assert_array_equal(run(A, B, packed, at, pitch, bias, relu=True), r(keep(S + bias)))
        np.testing.assert_array_equal(run(A, B, packed, at, pitch, bias, res, True), r(keep(r(S + bias) + res)))


# rows of every operand further apart than they are long (A by a part of a line, B by an odd number of values and from an odd
# value on, the residual by half a vector), in each kernel's range of K
@pytest.mark.parametrize('packed', [0, 1])
@pytest.mark.parametrize('M,N,K,lda,ldb,b_at,ldr,pitch', [
    (70001, 200, 56, 72, 203, 1, 204, 200), (70001, 201, 64, 128, 204, 2, 212, 203), (60001, 264, 128, 136, 265, 3, 268, 264), (140001, 7, 96, 104, 9, 1, 8, 7),
    (36399, 250, 200, 208, 251, 1, 252, 250), (20003, 1024, 256, 320, 1025, 5, 1028, 1024), (20003, 1000, 256, 264, 1000, 0, 1004, 1001)])
def test_strides(M, N, K, lda, ldb, b_at, ldr, pitch, packed):
    rng = np.random.default_rng(M + N + K)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    S = A @ B
    bias, res = whole(rng, N), whole(rng, (M, N))
    r, kw = E.round_bf16, dict(lda=lda, ldb=ldb, b_at=b_at, ldr=ldr)
    np.testing.assert_array_equal(run(A, B, packed, 0, pitch, bias, relu=True, **kw), r(np.maximum(S + bias, 0)))
    np.testing.assert_array_equal(run(A, B, packed, 0, pitch, bias, res, True, **kw), r(np.maximum(r(S + bias) + res, 0)))


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
    assert plan and 'streamed rows past B packed' in hk.describe(plan), hk.describe(plan)
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
    assert plan and 'streamed rows past B packed' in hk.describe(plan), hk.describe(plan)
    dX, dF, d1 = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (X, F, bias))
    dC, none = hk.DeviceBuffer(n * hw * hw * co * 2), hk.ptr_array([])
    hk.check(L.pml_hip_conv2d_invoke(plan, dX.ptr, dF.ptr, dC.ptr, d1.ptr, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    want = E.round_bf16(X.reshape(-1, ci) @ F.reshape(ci, co) + bias)
    np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (n * hw * hw, co))), want)
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('M,N,K,takes', [(25088, 128, 64, True), (19200, 128, 64, True), (17600, 128, 64, False), (8000, 200, 128, True), (12288, 128, 128, False), (25088, 128, 136, False)])
def test_which_rows_stream_past_a_right_hand_side_as_it_lies(M, N, K, takes):
    """Those that no direct tile takes, up to K = 128."""
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, K, N, N
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan
    text = hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    assert ('streamed rows past B as it lies' in text or 'or as it lies' in text) == takes, text
    assert takes or K > 128 or 'with B as it lies tile=' in text, text


# few rows and steps fewer than the device has wavefronts
@pytest.mark.parametrize('M,N,K', [(1374, 2000, 32), (4795, 511, 64), (8001, 200, 128), (9600, 251, 64)])
def test_few_steps(M, N, K):
    rng = np.random.default_rng(M)
    A, B, bias = whole(rng, (M, K)), whole(rng, (K, N)), whole(rng, N)
    np.testing.assert_array_equal(run(A, B, 0, bias=bias, relu=True), E.round_bf16(np.maximum(A @ B + bias, 0)))

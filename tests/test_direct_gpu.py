"""The direct tiles (csrc/direct.hip): 16 x 16 and 32 x 32 results per workgroup, eight wavefronts sharing its K, fragments
straight from memory.  Against float64 (int8: exact) where tiles, K steps and the
wavefronts' shares end raggedly."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
TILES = ['16x16w8', '32x32w8']


@pytest.fixture(scope='module', autouse=True)
def _device():
    hk.init(0)


def operands(kind, M, N, K, seed):
    rng = np.random.default_rng(seed)
    if kind == 'i8':
        return rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    return (E.round_bf16(A), E.round_bf16(B)) if kind == 'bf16' else (A, B)


def check(got, want, kind, K):
    # sums of K terms of size one: fp32 rounds every partial sum (at most sqrt(K) in size) to 2^-24, K of them in a row
    # at the very worst; a bf16 result is rounded once more, to 2^-9 of its value
    if kind == 'i8':
        np.testing.assert_array_equal(got, want)
    else:
        np.testing.assert_allclose(got, want, rtol=2.0 ** -8 if kind == 'bf16' else 1e-6, atol=2.0 ** -24 * K * np.sqrt(K) + 1e-6)


# one row; N odd (the right-hand side cannot be read as it lies), N a multiple of 4 and of 64; K of one chunk, of a partial
# step, of fewer steps than wavefronts, of one step more than whole shares; more tiles than CUs
SIZES = [(1, 1, 16), (1, 20, 32), (15, 17, 80), (16, 64, 512), (17, 68, 528), (33, 130, 1040), (49, 96, 2048), (70, 36, 272), (1000, 260, 48), (1000, 270, 80)]


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('tile', TILES + [None])
@pytest.mark.parametrize('M,N,K', SIZES)
def test_gemm(kind, tile, M, N, K, monkeypatch):
    if tile:
        monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile(tile))
    A, B = operands(kind, M, N, K, M + N + K)
    want = A.astype(np.float64) @ B.astype(np.float64)
    if kind == 'i8':
        check(T.run_gemm(A, B, hk.I8, hk.I32, invokes=2), want.astype(np.int64), kind, K)
    elif kind == 'f32':
        bias = np.linspace(-1, 1, N, dtype=np.float32)
        tail = hk.make_tail(ops=[(hk.EPI_RELU, hk.F32, 0, 0, 0.0)])
        got = T.run_gemm(A, B, hk.F32, hk.F32, init=bias, init_strides=(0, 1), init_dt=hk.F32, tail=tail)
        check(got, np.maximum(want + bias, 0), kind, K)
    else:
        res = E.round_bf16(np.random.default_rng(3).standard_normal((M, N)).astype(np.float32))
        tail = hk.make_tail(ops=[(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0)], operands=[(hk.BF16, N, 1)])
        got = E.bf16_from_bits(T.run_gemm(T.bf16(A), T.bf16(B), hk.BF16, hk.BF16, tail=tail, operands=[T.bf16(res)]))
        # (two roundings to bf16, the first of a sum of size sqrt(K))
        np.testing.assert_allclose(got, want + res, rtol=2.0 ** -8, atol=2.0 ** -8 * 4 * np.sqrt(K))


@pytest.mark.parametrize('tile', TILES)
def test_int8_requantised(tile, monkeypatch):
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile(tile))
    M, N, K = 37, 76, 336
    A, B = operands('i8', M, N, K, 5)
    scale = np.full(N, 2.0 ** -12, np.float32)
    tail = hk.make_tail(ops=[(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0),
                             (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -127.0), (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0),
                             (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)], operands=[(hk.F32, 0, 1)])
    got = T.run_gemm(A, B, hk.I8, hk.I32, c_dt=hk.I8, tail=tail, operands=[scale])
    v = np.clip((A.astype(np.int64) @ B.astype(np.int64)) / 4096.0, -127, 127)
    np.testing.assert_array_equal(got, (np.sign(v) * np.floor(np.abs(v) + 0.5)).astype(np.int8))


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('packed', [True, False])
@pytest.mark.parametrize('tile', TILES + [None, '64x64ks'])
@pytest.mark.parametrize('shape,k,co,stride', [((1, 7, 7, 64), 3, 48, 1), ((1, 7, 7, 512), 3, 96, 1), ((2, 9, 11, 96), 5, 40, 1), ((2, 9, 5, 16), 3, 20, 2), ((1, 14, 14, 80), 5, 33, 1), ((3, 6, 6, 32), 1, 64, 2)])
def test_conv(kind, tile, packed, shape, k, co, stride, monkeypatch):
    flags = hk.flag_conv(hk.CONV_IGEMM) | (hk.flag_tile(tile) if tile else 0)
    monkeypatch.setitem(T.FORCED, 'flags', flags)
    rng = np.random.default_rng(co)
    I, F = (rng.integers(-9, 10, s).astype(np.float32) for s in (shape, (k, k, shape[3], co)))  # exact sums in every type (fp32: below 2^24)
    dt, out, cast = {'f32': (hk.F32, hk.F32, lambda a: a), 'bf16': (hk.BF16, hk.BF16, T.bf16), 'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8))}[kind]
    got = T.run_conv(cast(I), cast(F), dt, out, stride=stride, packed=packed)
    n, h, w, _ = shape
    oh, ow = -(-h // stride), -(-w // stride)
    ph, pw = max(0, (oh - 1) * stride + k - h) // 2, max(0, (ow - 1) * stride + k - w) // 2
    pad = np.zeros((n, h + 2 * k, w + 2 * k, shape[3]))
    pad[:, ph:ph + h, pw:pw + w] = I
    want = sum(pad[:, y:y + (oh - 1) * stride + 1:stride, x:x + (ow - 1) * stride + 1:stride] @ F[y, x].astype(np.float64) for y in range(k) for x in range(k))
    if kind == 'bf16':
        np.testing.assert_array_equal(E.bf16_from_bits(got), E.round_bf16(want.astype(np.float32)))
    else:
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize('stride', [0, 2])
def test_two_products(stride):
    """A.B + A2.B2 over rows packed once: a wavefront's share of K begins in the first product and ends in the second."""
    rng = np.random.default_rng(21)
    OH, K1, K2, N = 7, 520, 264, 136
    M = OH * OH
    A, A2, B, B2 = (E.round_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((M, K1), (M, K2), (K1, N), (K2, N)))
    side = (OH - 1) * 2 + 1
    image = np.zeros((side, side, K2), np.float32)
    image[::2, ::2] = A2.reshape(OH, OH, K2)
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K1, K1, N, N
    d.k2, d.lda2, d.ldb2 = K2, K2, N
    if stride:
        d.a2_stride, d.a2_h, d.a2_w, d.a2_oh, d.a2_ow = stride, side, side, OH, OH
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan and 'wavefronts sharing K' in hk.describe(plan)
    dA, dB, dA2, dB2 = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, B, image if stride else A2, B2))
    dC, none = hk.DeviceBuffer(M * N * 2), hk.ptr_array([])
    hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr, None))
    hk.check(L.pml_hip_gemm_pack_b2(plan, dB2.ptr, None))
    hk.check(L.pml_hip_gemm_invoke2(plan, dA.ptr, None, dC.ptr, None, dA2.ptr, None, None, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    check(E.bf16_from_bits(dC.to_numpy(np.uint16, (M, N))), A.astype(np.float64) @ B + A2.astype(np.float64) @ B2, 'bf16', K1 + K2)
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('M,N,K', [(49, 512, 2048), (300, 72, 2064)])
def test_split_over_workgroups_by_name(kind, M, N, K, monkeypatch):
    """The two-launch split, which the direct tiles otherwise replace for most of these shapes."""
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile('64x64ks'))
    A, B = operands(kind, M, N, K, 9)
    dt, cast = {'f32': (hk.F32, lambda a: a), 'bf16': (hk.BF16, T.bf16), 'i8': (hk.I8, lambda a: a)}[kind]
    got = T.run_gemm(cast(A), cast(B), dt, hk.I32 if kind == 'i8' else dt, invokes=2)
    want = A.astype(np.float64) @ B.astype(np.float64)
    check(E.bf16_from_bits(got) if kind == 'bf16' else got, want, kind, K)


def held(desc, family='gemm', which=None):
    L = hk.lib()
    plan = L.pml_hip_conv2d_grad_dispatch(ctypes.byref(desc), which) if which is not None else getattr(L, 'pml_hip_%s_dispatch' % family)(ctypes.byref(desc))
    assert plan, L.pml_hip_last_error()
    return plan, L.pml_hip_plan_bytes(plan)


@pytest.mark.parametrize('kind,es', [('bf16', 2), ('i8', 1), ('f32', 4)])
def test_plans_hold_what_their_invokes_read(kind, es):
    """Workspaces of a split K only where no direct tile is taken: not for rows at hand, not for fp32, until the right-hand
    side is packed for the rest; right-hand sides of [K][N] for the transposed copy."""
    L, dt, N = hk.lib(), {'bf16': hk.BF16, 'i8': hk.I8, 'f32': hk.F32}[kind], 256
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = dt, hk.I32 if kind == 'i8' else dt, hk.I32 if kind == 'i8' else dt
    d.m, d.n, d.k = 196, N, 2048 if kind == 'i8' else 1024
    d.lda = d.ldb = d.k
    d.ldc, d.b_layout = N, 1
    plan, bytes_ = held(d)
    assert 'at hand tile=' in hk.describe(plan) and bytes_ == 0
    L.pml_hip_plan_free(plan)
    d.b_layout, d.ldb = 0, N
    plan, bytes_ = held(d)
    copy = N * d.k * es
    assert bytes_ == copy if kind == 'f32' else bytes_ > copy
    assert 'with B as it lies tile=' in hk.describe(plan)
    B = hk.DeviceBuffer(copy)
    hk.check(L.pml_hip_fill_u32(B.ptr, 0, copy // 4, None))
    hk.check(L.pml_hip_gemm_pack_b(plan, B.ptr, None))
    assert L.pml_hip_plan_bytes(plan) == copy
    L.pml_hip_plan_free(plan)


def conv(dt, n, hw, ci, co, k, stride):
    d = hk.Conv2dDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = dt
    o = (hw + stride - 1) // stride
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, hw, hw, ci, k, k, co, o, o
    d.stride_h = d.stride_w = stride
    d.dil_h = d.dil_w = 1
    d.pad_h = d.pad_w = max(0, (o - 1) * stride + k - hw) // 2
    return d


def test_convolution_plans_hold_what_their_invokes_read():
    for (hw, ci, co, k), split in (((28, 128, 128, 3), False), ((7, 512, 512, 3), True), ((56, 64, 64, 3), False)):
        plan, bytes_ = held(conv(hk.BF16, 1, hw, ci, co, k, 1), 'conv2d')
        filter_ = k * k * ci * co * 2
        assert bytes_ > filter_ if split else bytes_ == filter_, hk.describe(plan)
        hk.lib().pml_hip_plan_free(plan)
    # a data gradient: the flipped filter and the padded gradient of 70 channels; the columns of a stride of 2
    plan, bytes_ = held(conv(hk.BF16, 2, 14, 64, 70, 3, 1), which=0)
    assert bytes_ >= 9 * 64 * 72 * 2 + 2 * 14 * 14 * 72 * 2
    hk.lib().pml_hip_plan_free(plan)
    plan, bytes_ = held(conv(hk.F32, 2, 14, 64, 70, 3, 2), which=0)
    assert bytes_ >= 2 * 7 * 7 * 9 * 64 * 4
    hk.lib().pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind,out', [('f32', 'f32'), ('bf16', 'bf16'), ('bf16', 'f32'), ('i8', 'i32')])
@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('M,N,ldr,shift', [(33, 72, 72, 0), (17, 20, 28, 0), (1, 4, 4, 0), (33, 72, 72, 1), (17, 18, 18, 0), (40, 64, 70, 0)])
def test_tail_operands_read_ahead(kind, out, tile, M, N, ldr, shift):
    """A bias and a residual tensor, read before the sums exist where they are whole quads -- last rows and columns, rows of
    the residual longer than N -- and after them otherwise (a bias off its alignment, N or the residual's rows no multiple
    of four).  Whole numbers: every result is exact."""
    K = 80
    rng = np.random.default_rng(M + N + shift)
    A, B = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (K, N)).astype(np.float32)
    bias, res = rng.integers(-9, 10, N + shift).astype(np.float32), rng.integers(-9, 10, (M, ldr)).astype(np.float32)
    dts = {'f32': (hk.F32, lambda a: a, np.float32), 'bf16': (hk.BF16, T.bf16, np.uint16), 'i8': (hk.I8, lambda a: a.astype(np.int8), np.int8),
           'i32': (hk.I32, lambda a: a.astype(np.int32), np.int32)}
    (dt, cast, _), (odt, ocast, onp) = dts[kind], dts[out]
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, odt, odt, hk.flag_tile(tile)
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, K, N, N
    d.init_kind, d.init_dtype, d.init_col_stride = 1, odt, 1
    d.tail = hk.make_tail(ops=[(hk.EPI_ADD, odt, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_RELU, odt, 0, 0, 0.0)], operands=[(odt, ldr, 1)])
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, hk.lib().pml_hip_last_error()
    dA, dB, dI, dR = (hk.DeviceBuffer.from_numpy(x) for x in (cast(A), cast(B), ocast(bias), ocast(res)))
    es = np.dtype(onp).itemsize
    dC = hk.DeviceBuffer(M * N * es)
    hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, dB.ptr, dC.ptr, (dI.ptr.value if hasattr(dI.ptr, 'value') else dI.ptr) + shift * es,
                                          hk.ptr_array([dR.ptr]), hk.ptr_array([]), None))
    hk.check(hk.lib().pml_hip_stream_sync(None))
    got = dC.to_numpy(onp, (M, N))
    hk.lib().pml_hip_plan_free(plan)
    r = E.round_bf16 if out == 'bf16' else lambda a: a
    want = np.maximum(r(r(A @ B + bias[shift:]) + res[:, :N]), 0)
    np.testing.assert_array_equal(E.bf16_from_bits(got) if out == 'bf16' else got, want)


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('M,N,K,ldb,shift', [(1, 1, 16, 1, 0), (17, 67, 80, 67, 0), (33, 130, 272, 131, 1), (40, 65, 48, 66, 1), (5, 63, 1040, 67, 3), (20, 64, 80, 64, 1)])
def test_right_hand_side_rows_that_begin_anywhere(kind, tile, M, N, K, ldb, shift):
    """[K][N] read as it lies with N, the pitch and the pointer (`shift` elements off) no multiple of four: exact sums of whole
    numbers; the gap of the pitch holds NaNs / values that must not be read into a result; the buffer ends with the last row."""
    rng = np.random.default_rng(M + N + shift)
    top = 100 if kind == 'i8' else 4
    A, B = rng.integers(-top, top + 1, (M, K)).astype(np.float32), rng.integers(-top, top + 1, (K, N)).astype(np.float32)
    dt, out, cast, onp = {'f32': (hk.F32, hk.F32, lambda a: a.astype(np.float32), np.float32), 'bf16': (hk.BF16, hk.F32, T.bf16, np.float32),
                          'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8), np.int32)}[kind]
    flat = np.full(shift + (K - 1) * ldb + N, 77 if kind == 'i8' else np.nan, np.float32)
    for k in range(K):
        flat[shift + k * ldb:shift + k * ldb + N] = B[k]
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = dt, out, out
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, K, ldb, N
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan and 'with B as it lies' in hk.describe(plan), hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    d.flags = hk.flag_tile(tile)
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    dA, dB, dC = hk.DeviceBuffer.from_numpy(cast(A)), hk.DeviceBuffer.from_numpy(cast(flat)), hk.DeviceBuffer(M * N * 4)
    at = (dB.ptr.value if hasattr(dB.ptr, 'value') else dB.ptr) + shift * cast(flat).itemsize
    none = hk.ptr_array([])
    hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, at, dC.ptr, None, none, none, None))
    hk.check(hk.lib().pml_hip_stream_sync(None))
    np.testing.assert_array_equal(dC.to_numpy(onp, (M, N)), A @ B)
    hk.lib().pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind,M,N,K,split', [('bf16', 593, 606, 3808, True), ('bf16', 593, 606, 2816, True), ('bf16', 593, 606, 2800, False), ('f32x3', 650, 390, 2048, True), ('f32x3', 650, 390, 2016, False)])
def test_long_chains_of_some_tiles_are_split(kind, M, N, K, split):
    """More than 64 tiles: the K loop is shared out from the length on at which that pays."""
    if kind == 'f32x3':
        rng = np.random.default_rng(K)
        A, B = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    else:
        A, B = operands('bf16', M, N, K, K)
    d = hk.GemmDesc()
    dt = hk.F32 if kind == 'f32x3' else hk.BF16
    d.in_dtype = d.out_dtype = d.c_dtype = dt
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.flags = M, N, K, K, N, N, hk.FP32_AS_BF16X3 if kind == 'f32x3' else 0
    plan, _ = held(d)
    assert ('K split over workgroups' in hk.describe(plan)) == split, hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    want = A.astype(np.float64) @ B.astype(np.float64)
    if kind == 'f32x3':
        got = T.run_gemm(A, B, hk.F32, hk.F32, flags=hk.FP32_AS_BF16X3, invokes=2)
        assert np.abs(got - want).max() < 4 * 2.0 ** -16 * np.sqrt(K) * 0.25 + 1e-5
    else:
        check(E.bf16_from_bits(T.run_gemm(T.bf16(A), T.bf16(B), hk.BF16, hk.BF16, invokes=2)), want, 'bf16', K)


# columns on four and off it, K-rows of one 16-byte chunk, runs of taps, more taps than wavefronts; three channels: a patch matrix
# whose rows are padded, where a filter that does not end on a whole word is packed first
@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('shift', [0, 1])
@pytest.mark.parametrize('tile', TILES + [None])
@pytest.mark.parametrize('shape,k,co,stride', [((1, 9, 7, 32), 3, 48, 1), ((2, 7, 7, 16), 5, 33, 1), ((1, 8, 8, 96), 3, 131, 2), ((5, 6, 6, 64), 1, 66, 2),
                                               ((1, 9, 9, 3), 3, 33, 1), ((2, 8, 7, 3), 7, 20, 1), ((3, 5, 5, 5), 1, 17, 1)])
def test_filter_as_it_lies(kind, shift, tile, shape, k, co, stride):
    """A filter that comes with the call, `shift` elements into a buffer that ends with it and holds NaNs around it: exact sums
    of whole numbers, the same as over the packed filter; and again behind a filter of NaNs, which nothing may be kept of."""
    rng = np.random.default_rng(co + shift)
    n, h, w, ci = shape
    I, F = (rng.integers(-5, 6, s).astype(np.float32) for s in (shape, (k, k, ci, co)))
    dt, out, cast, onp = {'f32': (hk.F32, hk.F32, lambda a: a, np.float32), 'bf16': (hk.BF16, hk.F32, T.bf16, np.float32),
                          'i8': (hk.I8, hk.I32, lambda a: np.nan_to_num(a, nan=77).astype(np.int8), np.int32)}[kind]
    flat = np.full(shift + F.size + 8, np.nan, np.float32)
    flat[shift:shift + F.size] = F.ravel()
    oh, ow = -(-h // stride), -(-w // stride)
    d = hk.Conv2dDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = dt, out, out
    d.flags = hk.flag_conv(hk.CONV_IGEMM) | (hk.flag_tile(tile) if tile else 0)
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, w, ci, k, k, co, oh, ow
    d.stride_h = d.stride_w = stride
    d.dil_h = d.dil_w = 1
    d.pad_h, d.pad_w = max(0, (oh - 1) * stride + k - h) // 2, max(0, (ow - 1) * stride + k - w) // 2
    plans = [hk.lib().pml_hip_conv2d_dispatch(ctypes.byref(d)) for _ in range(2)]
    assert tile or 'with the filter as it lies tile=' in hk.describe(plans[0]), hk.describe(plans[0])
    dI, dF, dN, dO = hk.DeviceBuffer.from_numpy(cast(I)), hk.DeviceBuffer.from_numpy(cast(flat)), hk.DeviceBuffer.from_numpy(cast(np.full_like(flat, np.nan))), hk.DeviceBuffer(n * oh * ow * co * 4)
    dP = hk.DeviceBuffer.from_numpy(cast(F))
    none, at = hk.ptr_array([]), dF.ptr + shift * cast(flat).itemsize
    got = []
    for f in (at, dN.ptr, at):
        hk.check(hk.lib().pml_hip_conv2d_invoke(plans[0], dI.ptr, f, dO.ptr, None, none, none, None))
        got.append(dO.to_numpy(onp, (n, oh, ow, co)))
    hk.check(hk.lib().pml_hip_conv2d_pack_filter(plans[1], dP.ptr, None))
    hk.check(hk.lib().pml_hip_conv2d_invoke(plans[1], dI.ptr, None, dO.ptr, None, none, none, None))
    got.append(dO.to_numpy(onp, (n, oh, ow, co)))
    for p in plans:
        hk.lib().pml_hip_plan_free(p)
    pad = np.zeros((n, h + 2 * k, w + 2 * k, ci))
    pad[:, d.pad_h:d.pad_h + h, d.pad_w:d.pad_w + w] = I
    want = sum(pad[:, y:y + (oh - 1) * stride + 1:stride, x:x + (ow - 1) * stride + 1:stride] @ F[y, x].astype(np.float64) for y in range(k) for x in range(k))
    for g in (got[0], got[2], got[3]):
        np.testing.assert_array_equal(g, want)


@pytest.mark.parametrize('layout', [0, 1])
@pytest.mark.parametrize('M,N,K,plain', [(1, 17, 16, True), (7, 129, 208, True), (16, 26, 416, True), (100, 88, 272, True), (382, 253, 336, True),
                                         (2, 22, 3104, False), (1300, 700, 400, False)])
def test_split_fp32_of_few_results_is_plain_fp32(layout, M, N, K, plain):
    """fp32 that may be taken as three bf16 products: where direct tiles of fp32 MFMAs are faster the same bits as without the flag."""
    rng = np.random.default_rng(M + K)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K) if layout else (K, N)).astype(np.float32)
    dA, dB, dC = hk.DeviceBuffer.from_numpy(A), hk.DeviceBuffer.from_numpy(B), hk.DeviceBuffer(M * N * 4)
    got, none = [], hk.ptr_array([])
    for flags in (0, hk.FP32_AS_BF16X3):
        d = hk.GemmDesc()
        d.in_dtype = d.out_dtype = d.c_dtype = hk.F32
        d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = M, N, K, K, K if layout else N, N, layout, flags
        plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
        if flags and (plain or not layout):
            assert ('3 x f32' in hk.describe(plan)) != plain, hk.describe(plan)
        hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, dB.ptr, dC.ptr, None, none, none, None))
        got.append(dC.to_numpy(np.float32, (M, N)))
        hk.lib().pml_hip_plan_free(plan)
    if plain:
        np.testing.assert_array_equal(got[0], got[1])
    want = A.astype(np.float64) @ (B.T if layout else B).astype(np.float64)
    # (2^-16 of every product, at random; the largest of all results within 8 of its standard deviation sqrt(K))
    assert np.abs(got[1] - want).max() < 8 * 2.0 ** -16 * np.sqrt(K) + 1e-5


# 1 to 10 steps of K a wavefront, which two, three or four in flight share out, and 17; the last step whole, one vector and all but one
@pytest.mark.parametrize('M,N', [(5, 70), (37, 129)])
@pytest.mark.parametrize('K', [4, 128, 132, 256, 260, 380, 508, 640, 644, 768, 900, 1024, 1150 // 4 * 4, 1280, 2176])
def test_fp32_steps_in_flight(M, N, K):
    """The same bits from [K][N] as it lies as from [N][K], whatever the number of steps in flight; NaNs behind the operands."""
    A, B = operands('f32', M, N, K, M + K)
    pad = np.full(64, np.nan, np.float32)
    dA, dB, dBt = (hk.DeviceBuffer.from_numpy(np.concatenate([x.ravel(), pad])) for x in (A, B, np.ascontiguousarray(B.T)))
    dC, got, none = hk.DeviceBuffer(M * N * 4), [], hk.ptr_array([])
    for layout, b in ((0, dB), (1, dBt)):
        d = hk.GemmDesc()
        d.in_dtype = d.out_dtype = d.c_dtype = hk.F32
        d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = M, N, K, K, K if layout else N, N, layout, hk.flag_tile('16x16w8')
        plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
        hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, b.ptr, dC.ptr, None, none, none, None))
        got.append(dC.to_numpy(np.float32, (M, N)))
        hk.lib().pml_hip_plan_free(plan)
    check(got[0], A.astype(np.float64) @ B.astype(np.float64), 'f32', K)
    np.testing.assert_array_equal(got[0], got[1])


def test_which_kind_of_fp32_is_asked_of_sizes_alone():
    """Products that may be split, at every size either plain fp32 or three bf16 products from [K][N] and from [N][K], whatever the
    pitch: sizes where one layout's price is past the other's among them."""
    rng, kinds = np.random.default_rng(5), []
    sizes = [(2, 22, 3104), (556, 38, 1264), (36, 1896, 64)]
    sizes += [tuple(int(v) for v in np.exp(rng.uniform(np.log(lo), np.log(hi)))) for lo, hi in [((1, 16, 16), (1500, 1500, 4000))] * 250]
    for M, N, K in sizes:
        K = K // 4 * 4
        texts = []
        for layout, ldb in ((0, N), (0, N + 1), (0, N + 8), (1, K)):
            d = hk.GemmDesc()
            d.in_dtype = d.out_dtype = d.c_dtype = hk.F32
            d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = M, N, K, K, ldb, N, layout, hk.FP32_AS_BF16X3
            plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
            assert plan, hk.lib().pml_hip_last_error()
            texts.append('3 x f32' in hk.describe(plan))
            hk.lib().pml_hip_plan_free(plan)
        assert len(set(texts)) == 1, (M, N, K, texts)
        kinds.append(texts[0])
    assert 50 < sum(kinds) < 200  # (both kinds are met)


@pytest.mark.parametrize('M,N,K', [(251, 660, 848), (130, 2049, 80), (1250, 516, 64), (2048, 1024, 32), (2048, 2048, 32), (1030, 1990, 48), (60, 132, 1584)])
def test_fp32_tiles_agree_in_every_layout(M, N, K):
    """fp32 where direct tiles, tiles of 64 with K in two halves, plain ones and tiles of 128 meet: the same bits from B as it lies,
    packed and as [N][K]."""
    A, B = operands('f32', M, N, K, M + K)
    dA, dB, dBt, dC = hk.DeviceBuffer.from_numpy(A), hk.DeviceBuffer.from_numpy(B), hk.DeviceBuffer.from_numpy(np.ascontiguousarray(B.T)), hk.DeviceBuffer(M * N * 4)
    got, none = [], hk.ptr_array([])
    for form in ('kn', 'packed', 'nk'):
        d = hk.GemmDesc()
        d.in_dtype = d.out_dtype = d.c_dtype = hk.F32
        d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout = M, N, K, K, K if form == 'nk' else N, N, form == 'nk'
        plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
        print(hk.describe(plan), flush=True)
        if form == 'packed':
            hk.check(hk.lib().pml_hip_gemm_pack_b(plan, dB.ptr, None))
        hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, {'kn': dB.ptr, 'packed': None, 'nk': dBt.ptr}[form], dC.ptr, None, none, none, None))
        got.append(dC.to_numpy(np.float32, (M, N)))
        hk.lib().pml_hip_plan_free(plan)
    check(got[0], A.astype(np.float64) @ B.astype(np.float64), 'f32', K)
    np.testing.assert_array_equal(got[0], got[1])
    np.testing.assert_array_equal(got[0], got[2])

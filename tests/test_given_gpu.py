"""The 256 x 256 tile that reads a [K][N] right-hand side as it lies, through registers (csrc/given.hip).  Small whole numbers
make every sum exact, so every tail is compared value for value with numpy, where tiles, slabs and chunks of K end raggedly."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu

# one row, one chunk of K; four columns; rows, columns and K just below, at and above a tile / a slab / the ring's depth;
# N that ends inside a lane's sixteen columns; more tiles than CUs
SIZES = [(1, 4, 16), (255, 260, 48), (256, 256, 128), (257, 252, 144), (300, 64, 512), (129, 516, 640), (600, 1040, 1168), (4200, 4112, 80)]


@pytest.fixture(autouse=True)
def _tile(monkeypatch):
    hk.init(0)
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile('256x256w8'))


def whole(rng, shape):
    return rng.integers(-4, 5, shape).astype(np.float32)


@pytest.mark.parametrize('M,N,K', SIZES)
def test_bf16(M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    S = A @ B  # at most 16 K: exact
    bias, scale, shift, res = whole(rng, N), whole(rng, N), whole(rng, N), whole(rng, (M, N))
    r = E.round_bf16
    relu = (hk.EPI_RELU, hk.BF16, 0, 0, 0.0)
    kw = dict(init=T.bf16(bias), init_strides=(0, 1), init_dt=hk.BF16, invokes=2)

    def run(tail, operands=()):
        return E.bf16_from_bits(T.run_gemm(T.bf16(A), T.bf16(B), hk.BF16, hk.BF16, tail=tail, operands=[T.bf16(o) for o in operands], **kw))

    np.testing.assert_array_equal(run(hk.make_tail(ops=[relu])), r(np.maximum(S + bias, 0)))
    add = hk.make_tail(ops=[(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0), relu], operands=[(hk.BF16, N, 1)])
    np.testing.assert_array_equal(run(add, [res]), r(np.maximum(r(S + bias) + res, 0)))
    fold = hk.make_tail(ops=[(hk.EPI_MUL, hk.BF16, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 1, 0.0), relu],
                        operands=[(hk.BF16, 0, 1), (hk.BF16, 0, 1)])
    np.testing.assert_array_equal(run(fold, [scale, shift]), r(np.maximum(r(r(S + bias) * scale) + shift, 0)))
    steps = hk.make_tail(ops=[(hk.EPI_NEG, hk.BF16, 0, 0, 0.0), relu])  # (through LDS and the common tail)
    np.testing.assert_array_equal(run(steps), r(np.maximum(-r(S + bias), 0)))


def requant(n, with_sums):
    store = [(hk.EPI_STORE, hk.I32, 0, 0, 0.0)] if with_sums else []
    return hk.make_tail(ops=store + [(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0),
                                     (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -127.0), (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0),
                                     (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)], operands=[(hk.F32, 0, 1)])


@pytest.mark.parametrize('M,N,K', SIZES)
def test_int8(M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    S = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.int32)  # exact in float64
    np.testing.assert_array_equal(T.run_gemm(A, B, hk.I8, hk.I32, invokes=2), S)
    start = rng.integers(-1000, 1000, N, dtype=np.int32)
    scale = rng.uniform(0.5, 2, N).astype(np.float32) / np.float32(60 * np.sqrt(K))
    v = np.clip((S + start).astype(np.float32) * scale, -127, 127)
    want = np.trunc(v + np.copysign(np.float32(0.5), v)).astype(np.int8)
    kw = dict(init=start, init_strides=(0, 1), init_dt=hk.I32, operands=[scale], c_dt=hk.I8)
    np.testing.assert_array_equal(T.run_gemm(A, B, hk.I8, hk.I32, tail=requant(N, False), **kw), want)
    got, sums = T.run_gemm(A, B, hk.I8, hk.I32, tail=requant(N, True), extra_out=np.int32, **kw)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(sums, S + start)


@pytest.mark.parametrize('kind', ['bf16', 'i8'])
@pytest.mark.parametrize('n,ldb', [(260, 264), (260, 262), (258, 258)])
def test_packed_and_given_in_turn(kind, n, ldb):
    """A right-hand side packed once, ones that arrive with the call and are read as they lie, and ones that have to be turned
    (rows that are no multiple of four elements), which take the packed copy's place: each call multiplies what it was given."""
    M, K = 270, 272
    rng = np.random.default_rng(ldb)
    dt, out = (hk.BF16, hk.F32) if kind == 'bf16' else (hk.I8, hk.I32)
    A = whole(rng, (M, K))
    Bs = [whole(rng, (K, ldb)) for _ in range(2)]
    code = T.bf16 if kind == 'bf16' else lambda x: x.astype(np.int8)
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, out, out, T.FORCED['flags']
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, n, K, K, ldb, n
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, hk.lib().pml_hip_last_error()
    dA, dC = hk.DeviceBuffer.from_numpy(code(A)), hk.DeviceBuffer(M * n * 4)
    dB = [hk.DeviceBuffer.from_numpy(code(B)) for B in Bs]
    none = hk.ptr_array([])

    def call(b):
        hk.check(hk.lib().pml_hip_gemm_invoke(plan, dA.ptr, b, dC.ptr, None, none, none, None))
        hk.check(hk.lib().pml_hip_stream_sync(None))
        return dC.to_numpy(np.float32 if kind == 'bf16' else np.int32, (M, n)).astype(np.float32)

    want = [A @ B[:, :n] for B in Bs]
    np.testing.assert_array_equal(call(dB[0].ptr), want[0])
    hk.check(hk.lib().pml_hip_gemm_pack_b(plan, dB[1].ptr, None))
    np.testing.assert_array_equal(call(None), want[1])
    np.testing.assert_array_equal(call(dB[0].ptr), want[0])
    hk.check(hk.lib().pml_hip_gemm_pack_b(plan, dB[1].ptr, None))
    np.testing.assert_array_equal(call(None), want[1])
    hk.lib().pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind', ['bf16', 'i8'])
@pytest.mark.parametrize('M,N,K,lda,ldb,at', [(257, 260, 144, 160, 268, 4), (300, 64, 512, 528, 1000, 8), (129, 516, 640, 656, 520, 12)])
def test_strides(kind, M, N, K, lda, ldb, at):
    """Rows of A and B further apart than they are long, B on any four elements' boundary; the plan's text names the kernel."""
    rng = np.random.default_rng(M + N)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    code, es, dt, out, onp = (T.bf16, 2, hk.BF16, hk.F32, np.float32) if kind == 'bf16' else (lambda x: x.astype(np.int8), 1, hk.I8, hk.I32, np.int32)
    L = hk.lib()
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, out, out, T.FORCED['flags']
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, lda, ldb, N
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    want = 'with B as it lies or packed through registers mfma=f32_16x16x32_bf16' if kind == 'bf16' else 'with B as it lies through registers mfma=i32_16x16x64_i8'
    assert plan and want in hk.describe(plan), hk.describe(plan)
    wide_a, flat_b = np.full((M, lda), 99, np.float32), np.full(at + K * ldb, 99, np.float32)
    wide_a[:, :K] = A
    flat_b[at:].reshape(K, ldb)[:, :N] = B
    dA, dB, dC, none = hk.DeviceBuffer.from_numpy(code(wide_a)), hk.DeviceBuffer.from_numpy(code(flat_b)), hk.DeviceBuffer(M * N * 4), hk.ptr_array([])
    for b in (dB.ptr + at * es, None):
        if b is None:
            hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr + at * es, None))
        hk.check(L.pml_hip_fill_u32(dC.ptr, 0xdeadbeef, M * N, None))
        hk.check(L.pml_hip_gemm_invoke(plan, dA.ptr, b, dC.ptr, None, none, none, None))
        hk.check(L.pml_hip_stream_sync(None))
        np.testing.assert_array_equal(dC.to_numpy(onp, (M, N)), A @ B)
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind,K', [('i8', 64), ('i8', 16), ('bf16', 32), ('bf16', 8)])
@pytest.mark.parametrize('ldb', [26843544, 26843548, 30000000])
def test_rows_far_apart(kind, K, ldb):
    """Rows of B so far apart that the 80 bytes of K a slab's row offsets reach, more than K holds here, stay just below 2 GiB
    and do not: as it lies and through the transposed copy."""
    M, N = 70, 72
    rng = np.random.default_rng(K)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    code, es, dt, out = (T.bf16, 2, hk.BF16, hk.F32) if kind == 'bf16' else (lambda x: x.astype(np.int8), 1, hk.I8, hk.I32)
    ldb //= es
    L = hk.lib()
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, out, out, T.FORCED['flags']
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, K, ldb // 4 * 4, N
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    assert ('with B as it lies' in hk.describe(plan)) == (80 * d.ldb < 2 ** 31 if kind == 'i8' else 40 * d.ldb * 2 < 2 ** 31), hk.describe(plan)
    dA, dB, dC = hk.DeviceBuffer.from_numpy(code(A)), hk.DeviceBuffer(K * d.ldb * es), hk.DeviceBuffer(M * N * 4)
    rows = code(B)
    for k in range(K):
        hk.check(L.pml_hip_memcpy_h2d(dB.ptr + k * d.ldb * es, rows[k].ctypes.data, N * es, None))
    none = hk.ptr_array([])
    hk.check(L.pml_hip_gemm_invoke(plan, dA.ptr, dB.ptr, dC.ptr, None, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(plan)
    np.testing.assert_array_equal(dC.to_numpy(np.float32 if kind == 'bf16' else np.int32, (M, N)), A @ B)


def packed_product(kind, M, n, K, ldb, flags=0):
    """A plan with a right-hand side packed once, its operands and a call that returns the result's bytes."""
    rng = np.random.default_rng(M)
    L, dt = hk.lib(), hk.I8 if kind == 'i8' else hk.F32 if kind == 'f32x3' else hk.BF16
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, hk.I32 if kind == 'i8' else hk.F32, hk.I32 if kind == 'i8' else hk.F32, flags
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, n, K, K, ldb, n
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    codes = {hk.I8: np.arange(-4, 5).astype(np.int8), hk.F32: np.arange(-4, 5).astype(np.float32), hk.BF16: T.bf16(np.arange(-4, 5))}[dt]
    A, B = (hk.DeviceBuffer.from_numpy(codes[rng.integers(0, 9, s, np.uint8)]) for s in ((M, K), (K, ldb)))
    C, none = hk.DeviceBuffer(M * n * 4), hk.ptr_array([])
    hk.check(L.pml_hip_gemm_pack_b(plan, B.ptr, None))

    def call(b, c=C.ptr):
        hk.check(L.pml_hip_fill_u32(C.ptr, 0xdeadbeef, M * n, None))
        rc = L.pml_hip_gemm_invoke(plan, A.ptr, b, c, None, none, none, None)
        hk.check(L.pml_hip_stream_sync(None))
        return C.to_numpy(np.uint32, (M, n)) if rc == 0 else None

    return plan, B, call


@pytest.mark.parametrize('kind,K', [('bf16', 272), ('i8', 272), ('f32x3', 288)])
def test_a_refused_call_leaves_the_packed_copy(kind, K):
    """A call that brings a right-hand side the plan would have to turn, and is refused for another reason before that."""
    plan, B, call = packed_product(kind, 270, 260, K, 262, hk.flag_tile('64x64') | hk.FP32_AS_BF16X3 if kind == 'f32x3' else T.FORCED['flags'])
    want = call(None)
    assert call(B.ptr, None) is None
    np.testing.assert_array_equal(call(None), want)
    np.testing.assert_array_equal(call(B.ptr), want)
    np.testing.assert_array_equal(call(None), want)
    hk.lib().pml_hip_plan_free(plan)


def test_a_direct_tile_leaves_the_packed_copy():
    """Few rows, many columns: the right-hand side packed for the 256 x 256 tile, one that arrives with the call in rows this
    tile cannot read taken by a direct tile as it lies, and then the packed one again."""
    plan, B, call = packed_product('bf16', 256, 49152, 2560, 49154)
    assert '256x256' in hk.describe(plan) and 'with B as it lies tile=' in hk.describe(plan), hk.describe(plan)
    want = call(None)
    np.testing.assert_array_equal(call(B.ptr), want)
    np.testing.assert_array_equal(call(None), want)
    hk.lib().pml_hip_plan_free(plan)


def test_a_direct_tile_is_not_charged_a_copy_that_is_not_made():
    """256 rows, many columns: the direct tile of 32 x 64 would win only over a 256 x 256 tile that has its right-hand side
    transposed first; where that tile reads it as it lies, it runs."""
    for ldb, direct in ((49152, False), (49153, True)):
        d = hk.GemmDesc()
        d.in_dtype, d.out_dtype, d.c_dtype = hk.BF16, hk.F32, hk.F32
        d.m, d.n, d.k, d.lda, d.ldb, d.ldc = 256, 49152, 4096, 4096, ldb, 49152
        plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
        assert plan, hk.lib().pml_hip_last_error()
        text = hk.describe(plan)
        hk.lib().pml_hip_plan_free(plan)
        assert '256x256' in text and ('with B as it lies tile=' in text) == direct, text

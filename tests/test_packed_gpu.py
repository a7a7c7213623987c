"""Right-hand sides packed once behind every tile and element kind, products and convolutions.  Small whole numbers: every sum
is exact in every kind (fp32 as three bf16 products among them, whose packed form is heads and remainders)."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu

KINDS = {'f32': (hk.F32, hk.F32, lambda a: a, np.float32, 0), 'f32x3': (hk.F32, hk.F32, lambda a: a, np.float32, hk.FP32_AS_BF16X3),
         'bf16': (hk.BF16, hk.F32, T.bf16, np.float32, 0), 'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8), np.int32, 0)}


@pytest.fixture(autouse=True)
def _device():
    hk.init(0)


@pytest.mark.parametrize('kind', sorted(KINDS))
@pytest.mark.parametrize('tile', T.TILE_NAMES + ['16x16w8', '32x32w8'])
@pytest.mark.parametrize('M,N,K', [(300, 260, 288), (33, 65, 32), (70, 130, 1184)])
def test_product(kind, tile, M, N, K):
    dt, out, cast, onp, flags = KINDS[kind]
    rng = np.random.default_rng(M)
    A, B = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (K, N)))
    d = hk.GemmDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, out, out, flags | hk.flag_tile(tile)
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = M, N, K, K, N, N
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    dA, dB, dC, none = hk.DeviceBuffer.from_numpy(cast(A)), hk.DeviceBuffer.from_numpy(cast(B)), hk.DeviceBuffer(M * N * 4), hk.ptr_array([])
    hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr, None))
    for _ in range(2):
        hk.check(L.pml_hip_fill_u32(dC.ptr, 0xdeadbeef, M * N, None))
        hk.check(L.pml_hip_gemm_invoke(plan, dA.ptr, None, dC.ptr, None, none, none, None))
        hk.check(L.pml_hip_stream_sync(None))
        np.testing.assert_array_equal(dC.to_numpy(onp, (M, N)), A @ B)
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('kind', sorted(KINDS))
@pytest.mark.parametrize('tile', T.TILE_NAMES)
@pytest.mark.parametrize('shape,k,co,stride', [((2, 13, 11, 32), 3, 136, 1), ((1, 9, 17, 96), 3, 72, 2)])
def test_convolution(kind, tile, shape, k, co, stride, monkeypatch):
    dt, out, cast, _, flags = KINDS[kind]
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_conv(hk.CONV_IGEMM) | hk.flag_tile(tile))
    rng = np.random.default_rng(co)
    I, F = (rng.integers(-4, 5, s).astype(np.float32) for s in (shape, (k, k, shape[3], co)))
    got = T.run_conv(cast(I), cast(F), dt, out, stride=stride, packed=True, flags=flags)
    n, h, w, ci = shape
    oh, ow = -(-h // stride), -(-w // stride)
    ph, pw = max(0, (oh - 1) * stride + k - h) // 2, max(0, (ow - 1) * stride + k - w) // 2
    pad = np.zeros((n, h + 2 * k, w + 2 * k, ci), np.float32)
    pad[:, ph:ph + h, pw:pw + w] = I
    want = sum(pad[:, y:y + (oh - 1) * stride + 1:stride, x:x + (ow - 1) * stride + 1:stride] @ F[y, x] for y in range(k) for x in range(k))
    np.testing.assert_array_equal(got, want)


def two_products(m, n, k, k2, lda2=None, ldb2=None, pixels=None, layout=0):
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout = m, n, k, k, k if layout else n, n, layout
    d.k2, d.lda2, d.ldb2 = k2, lda2 or k2, ldb2 or (k2 if layout else n)
    if pixels:
        d.a2_stride, d.a2_h, d.a2_w, d.a2_oh, d.a2_ow = pixels
    return d


@pytest.mark.parametrize('tile', [None, '64x64', '32x32w8'])
@pytest.mark.parametrize('desc', [dict(lda2=1 << 30), dict(pixels=(1, 1, 2, 1, 2), lda2=1 << 30), dict(ldb2=1 << 30, layout=1), dict(pixels=(2, 3, 1, 2, 1), lda2=1 << 29)])
def test_second_product_of_two_gib_is_refused(desc, tile):
    """Offsets into its operands are 32 bits below 2 GiB, as the first product's are (the rows that would be read lie at 2 GiB
    exactly: nothing is read where they are not refused either)."""
    d = two_products(2, 16, 16, 16, **desc)
    if tile:
        d.flags = hk.flag_tile(tile)
    if desc.get('layout'):
        d.n = 2
        d.ldc = 16
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    buf, none = hk.DeviceBuffer(4096), hk.ptr_array([])
    hk.check(L.pml_hip_fill_u32(buf.ptr, 0, 1024, None))
    assert L.pml_hip_gemm_invoke2(plan, buf.ptr, buf.ptr, buf.ptr, None, buf.ptr, buf.ptr, None, none, none, None) != 0
    L.pml_hip_plan_free(plan)


@pytest.mark.parametrize('stride', [0, 2])
def test_second_product_up_to_two_gib(stride):
    """The last row read ends just below 2 GiB."""
    rng = np.random.default_rng(stride)
    K, K2, N = 16, 24, 20
    A, B, B2 = (rng.integers(-4, 5, s).astype(np.float32) for s in ((2, K), (K, N), (K2, N)))
    A2 = rng.integers(-4, 5, (2, K2)).astype(np.float32)
    rows = 2 if stride else 1  # between the two rows read
    lda2 = ((1 << 30) - 32) // rows // 8 * 8
    d = two_products(2, N, K, K2, lda2=lda2, pixels=(2, 1, 3, 1, 2) if stride else None)
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    dA, dB, dB2, dC, none = (hk.DeviceBuffer.from_numpy(T.bf16(A)), hk.DeviceBuffer.from_numpy(T.bf16(B)), hk.DeviceBuffer.from_numpy(T.bf16(B2)),
                             hk.DeviceBuffer(2 * N * 2), hk.ptr_array([]))
    dA2 = hk.DeviceBuffer(2 << 30)
    bits = T.bf16(A2)
    for i in range(2):
        hk.check(L.pml_hip_memcpy_h2d(dA2.ptr + i * rows * lda2 * 2, bits[i].ctypes.data, K2 * 2, None))
    hk.check(L.pml_hip_gemm_invoke2(plan, dA.ptr, dB.ptr, dC.ptr, None, dA2.ptr, dB2.ptr, None, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(plan)
    np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (2, N))), E.round_bf16(A @ B + A2 @ B2))


@pytest.mark.parametrize('form', ['packed', 'given', 'rows'])
@pytest.mark.parametrize('stride', [0, 2])
@pytest.mark.parametrize('tile', T.TILE_NAMES + ['16x16w8', '32x32w8', None])
def test_two_products(tile, stride, form):
    """Both right-hand sides packed once, as [K][N] with the call, and as [N][K]: slabs of both products behind one another, shared
    out among workgroups where K is split, from the middle of either on."""
    rng = np.random.default_rng(stride)
    K, K2, N, side = 1096, 648, 72, 6
    M = side * side
    A, A2, B, B2 = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (M, K2), (K, N), (K2, N)))
    b1, b2 = (rng.integers(-9, 10, N).astype(np.float32) for _ in range(2))
    wide = (side - 1) * 2 + 1
    image = np.zeros((wide, wide, K2), np.float32)
    image[::2, ::2] = A2.reshape(side, side, K2)
    d = two_products(M, N, K, K2, pixels=(stride, wide, wide, side, side) if stride else None, layout=int(form == 'rows'))
    d.out_dtype = d.c_dtype = d.init_dtype = hk.F32
    d.init_kind = d.init_col_stride = d.init2_kind = 1
    d.flags = hk.flag_tile(tile) if tile else 0
    L = hk.lib()
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    turned = (lambda x: np.ascontiguousarray(x.T)) if form == 'rows' else lambda x: x
    dA, dB, dA2, dB2 = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, turned(B), image if stride else A2, turned(B2)))
    d1, d2, dC, none = hk.DeviceBuffer.from_numpy(b1), hk.DeviceBuffer.from_numpy(b2), hk.DeviceBuffer(M * N * 4), hk.ptr_array([])
    if form == 'packed':
        hk.check(L.pml_hip_gemm_pack_b(plan, dB.ptr, None))
        hk.check(L.pml_hip_gemm_pack_b2(plan, dB2.ptr, None))
    given = (None, None) if form == 'packed' else (dB.ptr, dB2.ptr)
    for _ in range(2):
        hk.check(L.pml_hip_fill_u32(dC.ptr, 0xdeadbeef, M * N, None))
        hk.check(L.pml_hip_gemm_invoke2(plan, dA.ptr, given[0], dC.ptr, d1.ptr, dA2.ptr, given[1], d2.ptr, none, none, None))
        hk.check(L.pml_hip_stream_sync(None))
        np.testing.assert_array_equal(dC.to_numpy(np.float32, (M, N)), A @ B + A2 @ B2 + b1 + b2)
    L.pml_hip_plan_free(plan)

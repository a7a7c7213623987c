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

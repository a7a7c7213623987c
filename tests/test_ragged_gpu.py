"""Tails of products and convolutions whose last columns are no whole quad and whose rows begin anywhere (csrc/igemm_tail.h):
whole numbers, so that every tail is compared value for value with numpy, through tiles whose sums pass through LDS."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
TILES = ['64x64', '128x128w8s2', '256x256w8', '64x64ks', '16x16w8', '32x32w8']


@pytest.fixture(autouse=True)
def _device():
    hk.init(0)


def whole(rng, shape, top=4):
    return rng.integers(-top, top + 1, shape).astype(np.float32)


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('kind', ['f32', 'bf16'])
@pytest.mark.parametrize('M,N', [(1, 1), (67, 2), (130, 35), (70, 131), (33, 66)])
def test_float_tails(kind, tile, M, N, monkeypatch):
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile(tile))
    K = 1168 if tile == '64x64ks' else 144
    dt, cast, back, r = (hk.BF16, T.bf16, E.bf16_from_bits, E.round_bf16) if kind == 'bf16' else (hk.F32, lambda a: a, lambda a: a, lambda a: a)
    rng = np.random.default_rng(M + N)
    A, B = whole(rng, (M, K)), whole(rng, (K, N))
    bias, x, y = whole(rng, N), whole(rng, N), whole(rng, N)
    S = A @ B + bias
    relu = (hk.EPI_RELU, dt, 0, 0, 0.0)

    def run(tail, operands=(), init=bias, strides=(0, 1)):
        return back(T.run_gemm(cast(A), cast(B), dt, dt, init=cast(init), init_strides=strides, init_dt=dt, tail=tail,
                               operands=[cast(o) for o in operands], invokes=2))

    np.testing.assert_array_equal(run(hk.make_tail(ops=[relu])), np.maximum(r(S), 0))
    rows = whole(rng, M)
    np.testing.assert_array_equal(run(hk.make_tail(ops=[relu]), init=rows, strides=(1, 0)), np.maximum(r(A @ B + rows[:, None]), 0))
    ldr = (N + 3) // 4 * 4
    res = whole(rng, (M, ldr))
    add = hk.make_tail(ops=[(hk.EPI_ADD, dt, hk.OPND_TENSOR, 0, 0.0), relu], operands=[(dt, ldr, 1)])
    np.testing.assert_array_equal(run(add, [res]), np.maximum(r(r(S) + res[:, :N]), 0))
    steps = hk.make_tail(ops=[(hk.EPI_MUL, dt, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_SUB, dt, hk.OPND_TENSOR, 1, 0.0), (hk.EPI_MIN, dt, hk.OPND_IMM, 0, 96.0)],
                         operands=[(dt, 0, 1), (dt, 0, 1)])
    np.testing.assert_array_equal(run(steps, [x, y]), np.minimum(r(r(r(S) * x) - y), 96))


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('M,N', [(1, 1), (67, 2), (130, 35), (70, 131), (33, 66)])
def test_int8_tails(tile, M, N, monkeypatch):
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile(tile))
    K = 2320 if tile == '64x64ks' else 144
    rng = np.random.default_rng(M + N)
    A, B = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    S = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.int32)
    start = rng.integers(-1000, 1000, N, dtype=np.int32)
    kw = dict(init=start, init_strides=(0, 1), init_dt=hk.I32)
    relu = hk.make_tail(ops=[(hk.EPI_RELU, hk.I32, 0, 0, 0.0)])
    np.testing.assert_array_equal(T.run_gemm(A, B, hk.I8, hk.I32, tail=relu, invokes=2, **kw), np.maximum(S + start, 0))
    for scale, cs in ((rng.uniform(0.5, 2, N).astype(np.float32) / np.float32(60 * np.sqrt(K)), 1), (np.full(1, 0.001, np.float32), 0)):
        v = np.clip((S + start).astype(np.float32) * scale, -127, 127)
        want = np.trunc(v + np.copysign(np.float32(0.5), v)).astype(np.int8)
        for sums in (False, True):
            store = [(hk.EPI_STORE, hk.I32, 0, 0, 0.0)] if sums else []
            tail = hk.make_tail(ops=store + [(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0),
                                             (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -127.0), (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0),
                                             (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)], operands=[(hk.F32, 0, cs)])
            got = T.run_gemm(A, B, hk.I8, hk.I32, tail=tail, operands=[scale], c_dt=hk.I8, extra_out=np.int32 if sums else None, **kw)
            if sums:
                got, stored = got
                np.testing.assert_array_equal(stored, S + start)
            np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('tile', ['64x64', '128x128w8s2', '64x64ks', '16x16w8', '32x32w8'])
@pytest.mark.parametrize('shape,kh,kw,co,stride', [((2, 5, 3, 16), 7, 7, 20, 1), ((1, 12, 9, 48), 5, 5, 70, 2), ((1, 6, 17, 112), 3, 3, 33, 1), ((3, 9, 10, 32), 1, 5, 64, 1)])
def test_filter_rows_as_one_tap(kind, tile, shape, kh, kw, co, stride, monkeypatch):
    """Pixels of less than a slab (or of a broken number of them): the taps of a filter row are one run over neighbouring
    pixels, whose chunks lie inside or outside the image one by one -- images narrower than the filter among them."""
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_conv(hk.CONV_IGEMM) | hk.flag_tile(tile))
    rng = np.random.default_rng(co)
    n, h, w, ci = shape
    I, F = whole(rng, shape), whole(rng, (kh, kw, ci, co))  # sums below 2^24
    dt, out, cast = {'f32': (hk.F32, hk.F32, lambda a: a), 'bf16': (hk.BF16, hk.BF16, T.bf16), 'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8))}[kind]
    got = T.run_conv(cast(I), cast(F), dt, out, stride=stride)
    oh, ow = -(-h // stride), -(-w // stride)
    ph, pw = max(0, (oh - 1) * stride + kh - h) // 2, max(0, (ow - 1) * stride + kw - w) // 2
    pad = np.zeros((n, h + 2 * kh, w + 2 * kw, ci))
    pad[:, ph:ph + h, pw:pw + w] = I
    want = sum(pad[:, y:y + (oh - 1) * stride + 1:stride, x:x + (ow - 1) * stride + 1:stride] @ F[y, x].astype(np.float64) for y in range(kh) for x in range(kw))
    np.testing.assert_array_equal(E.bf16_from_bits(got) if kind == 'bf16' else got, E.round_bf16(want.astype(np.float32)) if kind == 'bf16' else want)


@pytest.mark.parametrize('kind', ['f32', 'f32x3', 'bf16', 'i8'])
@pytest.mark.parametrize('packed', [False, True])
@pytest.mark.parametrize('tile', [None, '64x64', '128x128w8', '64x64ks', '32x32w8'])
@pytest.mark.parametrize('shape,kh,kw,co,stride,dil', [((2, 9, 5, 16), 5, 3, 20, 1, 2), ((1, 13, 9, 48), 3, 5, 70, 2, 3), ((1, 8, 11, 112), 2, 3, 33, 1, 4)])
def test_filter_rows_as_one_tap_dilated(kind, packed, tile, shape, kh, kw, co, stride, dil):
    """The same with filter rows further apart (the taps of a row stay neighbours), fp32 as three bf16 products among the kinds,
    where every value counts as whole numbers do; filters that arrive with the call and packed ones."""
    rng = np.random.default_rng(co + dil)
    n, h, w, ci = shape
    I, F = whole(rng, shape), whole(rng, (kh, kw, ci, co))
    dt, out, cast, onp = {'f32': (hk.F32, hk.F32, lambda a: a, np.float32), 'f32x3': (hk.F32, hk.F32, lambda a: a, np.float32), 'bf16': (hk.BF16, hk.F32, T.bf16, np.float32),
                          'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8), np.int32)}[kind]
    d = hk.Conv2dDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = dt, out, out
    d.flags = hk.flag_conv(hk.CONV_IGEMM) | (hk.flag_tile(tile) if tile else 0) | (hk.FP32_AS_BF16X3 if kind == 'f32x3' else 0)
    ph, pw = (kh - 1) * dil // 2, (kw - 1) // 2
    oh, ow = (h + 2 * ph - (kh - 1) * dil - 1) // stride + 1, (w + 2 * pw - kw) // stride + 1
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, w, ci, kh, kw, co, oh, ow
    d.stride_h = d.stride_w = stride
    d.dil_h, d.dil_w, d.pad_h, d.pad_w = dil, 1, ph, pw
    L = hk.lib()
    plan = L.pml_hip_conv2d_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    dI, dF, dO, none = hk.DeviceBuffer.from_numpy(cast(I)), hk.DeviceBuffer.from_numpy(cast(F)), hk.DeviceBuffer(n * oh * ow * co * 4), hk.ptr_array([])
    if packed:
        hk.check(L.pml_hip_conv2d_pack_filter(plan, dF.ptr, None))
    hk.check(L.pml_hip_conv2d_invoke(plan, dI.ptr, None if packed else dF.ptr, dO.ptr, None, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(plan)
    pad = np.zeros((n, h + 2 * ph, w + 2 * pw, ci))
    pad[:, ph:ph + h, pw:pw + w] = I
    want = sum(pad[:, y * dil:y * dil + (oh - 1) * stride + 1:stride, x:x + (ow - 1) * stride + 1:stride] @ F[y, x].astype(np.float64) for y in range(kh) for x in range(kw))
    np.testing.assert_array_equal(dO.to_numpy(onp, (n, oh, ow, co)), want)

"""Tails of products and convolutions whose last columns are no whole quad and whose rows begin anywhere (csrc/igemm_tail.h):
whole numbers, so that every tail is compared value for value with numpy, through tiles whose sums pass through LDS."""
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

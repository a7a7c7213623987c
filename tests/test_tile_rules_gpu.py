"""Which products take 64 x 64 tiles, and which of those share K in two wavefront grids: by the tail and by what else a tile waits for."""
import ctypes

import numpy as np
import pytest

from plaidml_amd import edsl as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
SHARED, PLAIN = 'tile=64x64 (8 wavefronts, K split in two) ', 'tile=64x64 '


def run(kind, m, n, k, tail='relu', k2=0, tile=None):
    """C, what it should be, by how much it may differ and the plan's text; operands from the sizes alone."""
    L, rng, f32 = hk.lib(), np.random.default_rng(m + n + k), kind == 'f32'
    dt, cast = (hk.F32, lambda a: a) if f32 else (hk.BF16, E.to_bf16_bits)
    draw = lambda *s: E.round_bf16(rng.standard_normal(s).astype(np.float32))  # noqa: E731
    A, B, A2, B2, b, b2, R, S = draw(m, k), draw(k, n), draw(m, max(k2, 1)), draw(max(k2, 1), n), draw(n), draw(n), draw(m, n), draw(n)
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = dt
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = m, n, k, k, n, n
    d.init_kind, d.init_dtype, d.init_row_stride, d.init_col_stride = 1, dt, 0, 1
    relu, operands, values = (hk.EPI_RELU, dt, 0, 0, 0.0), [], []
    want = A.astype(np.float64) @ B + b
    if k2:
        want = want + A2.astype(np.float64) @ B2 + b2
    # t exact products of size one: a rounding each, 2^-24 of a partial sum of up to 4 sqrt(t)
    size, off = np.abs(want), np.full_like(want, 4 * (k + k2) ** 1.5 * 2.0 ** -24)
    if tail == 'relu':
        ops = [relu]
    elif tail == 'residual':
        ops, operands, values = [(hk.EPI_ADD, dt, hk.OPND_TENSOR, 0, 0.0), relu], [(dt, n, 1)], [R]
        want, size = want + R, size + np.abs(R)
    else:
        ops, operands, values = [(hk.EPI_MUL, dt, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_ADD, dt, hk.OPND_TENSOR, 1, 0.0), relu], [(dt, 0, 1), (dt, 0, 1)], [S, b2]
        want, size, off = want * S + b2, size * np.abs(S) + np.abs(b2), off * np.abs(S)
    d.tail = hk.make_tail(ops=ops, operands=operands)
    if k2:
        d.k2, d.lda2, d.ldb2, d.init2_kind = k2, k2, n, 1
    d.flags = hk.flag_tile(tile) if tile else 0
    plan = L.pml_hip_gemm_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    text = hk.describe(plan)
    dev = [hk.DeviceBuffer.from_numpy(cast(x)) for x in (A, B, b, A2, B2, b2)]
    held = [hk.DeviceBuffer.from_numpy(cast(x)) for x in values]
    out, none, at = hk.DeviceBuffer(m * n * (4 if f32 else 2)), hk.ptr_array([]), hk.ptr_array([x.ptr for x in held])
    if k2:
        hk.check(L.pml_hip_gemm_pack_b2(plan, dev[4].ptr, None))
        hk.check(L.pml_hip_gemm_invoke2(plan, dev[0].ptr, dev[1].ptr, out.ptr, dev[2].ptr, dev[3].ptr, None, dev[5].ptr, at, none, None))
    else:
        hk.check(L.pml_hip_gemm_invoke(plan, dev[0].ptr, dev[1].ptr, out.ptr, dev[2].ptr, at, none, None))
    got = out.to_numpy(np.float32 if f32 else np.uint16, (m, n))
    L.pml_hip_plan_free(plan)
    # ... and up to three roundings of what is `size` large on the way, to 8 or 24 bits
    return got if f32 else E.from_bf16_bits(got), np.maximum(want, 0), off + 4 * size * (2.0 ** -24 if f32 else 2.0 ** -8), text


# a network's layer at batch 1, few columns, one tile, a K that two grids share whatever the tail
@pytest.mark.parametrize('m,n,k,k2,shared', [(784, 512, 128, 256, False), (2831, 72, 32, 96, False), (3400, 64, 64, 32, False), (1281, 520, 128, 128, False),
                                             (2000, 520, 512, 512, True)])
def test_two_products(m, n, k, k2, shared):
    """A second product and its start values are waited for: short K's of two products are not shared."""
    got, want, bound, text = run('bf16', m, n, k, k2=k2)
    assert (SHARED if shared else PLAIN) in text and ('K split in two' in text) == shared, text
    named = run('bf16', m, n, k, k2=k2, tile='64x64w8k2' if shared else '64x64')[0]
    np.testing.assert_array_equal(got, named)
    assert (np.abs(got - want) <= bound).all()


# 900 tiles of 64 x 64 and 225 of 128 x 128, 754 and 195, the last 768; rows off 16 bytes; a K of three slabs
@pytest.mark.parametrize('m,n,k,tail,k2,large', [(3162, 1144, 120, 'scale', 0, True), (3162, 1144, 120, 'relu', 0, True), (3162, 1144, 120, 'residual', 0, False),
                                                 (3162, 1146, 120, 'scale', 0, False), (1799, 1648, 80, 'scale', 0, False), (1536, 2048, 128, 'scale', 0, False),
                                                 (1537, 2040, 128, 'scale', 0, True), (1799, 1648, 136, 'scale', 0, True), (1799, 1648, 32, 'relu', 48, True)])
def test_two_slabs_and_less(m, n, k, tail, k2, large):
    """128 x 128 tiles of a short K: where tiles of 64 would be more than three a CU, but for residuals and rows off 16 bytes, and
    under two products."""
    got, want, bound, text = run('bf16', m, n, k, tail, k2)
    assert ('tile=128x128 (8 wavefronts)' if large else PLAIN) in text, text
    named = run('bf16', m, n, k, tail, k2, tile='128x128w8' if large else '64x64')[0]
    for c in (got, named):
        assert (np.abs(c - want) <= bound).all()


# fp32, K of less than 2 KB: 264 tiles and 256 of them, rows off 16 bytes; a longer K
@pytest.mark.parametrize('m,n,k,tail,shared', [(1381, 768, 120, 'scale', False), (1381, 768, 120, 'residual', True), (1381, 768, 120, 'relu', True), (1024, 1024, 120, 'scale', True),
                                               (1381, 766, 120, 'scale', True), (1381, 768, 512, 'scale', True)])
def test_fp32_under_scale_and_shift(m, n, k, tail, shared):
    got, want, bound, text = run('f32', m, n, k, tail)
    assert (SHARED if shared else PLAIN) in text and ('K split in two' in text) == shared, text
    named = run('f32', m, n, k, tail, tile='64x64w8k2' if shared else '64x64')[0]
    np.testing.assert_array_equal(got, named)
    assert (np.abs(got - want) <= bound).all()


def text_of(kind, m, n, k, layout=0, flags=0):
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = kind
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = m, n, k, k, k if layout else n, n, layout, flags
    plan = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(d))
    text = hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    return text


# one slab over 1.78 and 1.59 rounds of 128 x 128; a round less than half full; edges that cost the large tiles more; two slabs
@pytest.mark.parametrize('m,n,k,large', [(7295, 944, 12, True), (4690, 1308, 28, True), (9911, 400, 12, False), (50809, 272, 28, False), (7295, 944, 36, False)])
def test_fp32_of_one_slab(m, n, k, large):
    assert ('tile=128x128 (8 wavefronts, 2 stages) ' if large else PLAIN) in text_of(hk.F32, m, n, k)


@pytest.mark.parametrize('layout', [0, 1])
@pytest.mark.parametrize('m,n,k,direct', [(6, 59, 4000, False), (120, 71, 2688, False), (1030, 36, 2608, True), (2, 37, 3500, True), (6, 59, 1200, True)])
def test_fp32_of_a_long_k_and_few_columns(m, n, k, direct, layout):
    """Split in both layouts where a direct tile loses more over [K][N] than it gains over rows of K."""
    text = text_of(hk.F32, m, n, k, layout)
    assert ('with rows of K at hand' in text) == direct and ('with B as it lies' in text) == (direct and not layout), text


@pytest.mark.parametrize('layout', [0, 1])
@pytest.mark.parametrize('m,n,k,split', [(29, 3872, 96, True), (34, 2320, 96, True), (40, 1800, 200, False), (16, 3872, 96, False),
                                         (191, 381, 64, False), (177, 300, 64, False), (5, 27, 1040, False), (4, 36, 2192, True)])
def test_split_fp32_of_two_rounds(m, n, k, split, layout):
    assert ('3 x f32' in text_of(hk.F32, m, n, k, layout, hk.FP32_AS_BF16X3)) == split


# 7 x 7 taps of 40 channels, 4 KB of K; odd columns, a residual over them; the same in int8 and of fewer channels
@pytest.mark.parametrize('kind,out,ci,co,residual,lies', [(hk.BF16, hk.BF16, 40, 16, False, False), (hk.BF16, hk.BF16, 40, 15, False, True),
                                                          (hk.BF16, hk.BF16, 40, 15, True, False), (hk.I8, hk.I32, 32, 16, False, True),
                                                          (hk.BF16, hk.BF16, 16, 16, False, True)])
def test_filters_of_a_long_k_that_come_with_the_call(kind, out, ci, co, residual, lies):
    d = hk.Conv2dDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = kind, out, out
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = 1, 74, 18, ci, 7, 7, co, 74, 18
    d.stride_h = d.stride_w = d.dil_h = d.dil_w = 1
    d.pad_h = d.pad_w = 3
    if residual:
        d.tail = hk.make_tail(ops=[(hk.EPI_ADD, out, hk.OPND_TENSOR, 0, 0.0)], operands=[(out, co, 1)])
    plan = hk.lib().pml_hip_conv2d_dispatch(ctypes.byref(d))
    assert ('with the filter as it lies' in hk.describe(plan)) == lies, hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)


# int8 of 3 KB of K: ten rows of tiles of 32, and fewer channels; fp32 of a long K in eight rounds of 16 x 16 and in less than one
@pytest.mark.parametrize('kind,out,n,h,ci,k,stride,co,text', [(hk.I8, hk.I32, 4, 20, 64, 7, 2, 12, None), (hk.I8, hk.I32, 4, 20, 16, 3, 2, 12, 'with the filter as it lies'),
                                                             (hk.F32, hk.F32, 7, 68, 128, 3, 1, 11, 'over its window in LDS'),
                                                             (hk.I8, hk.I32, 4, 20, 96, 5, 2, 48, 'with the filter as it lies'),
                                                             (hk.F32, hk.F32, 1, 14, 128, 3, 1, 11, 'direct tile=16x16')])
def test_convolutions_beside_their_direct_tiles(kind, out, n, h, ci, k, stride, co, text):
    d = hk.Conv2dDesc()
    d.in_dtype, d.out_dtype, d.c_dtype = kind, out, out
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, h, ci, k, k, co, -(-h // stride), -(-h // stride)
    d.stride_h = d.stride_w = stride
    d.dil_h = d.dil_w = 1
    d.pad_h = d.pad_w = k // 2
    plan = hk.lib().pml_hip_conv2d_dispatch(ctypes.byref(d))
    got = hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    assert text in got if text else 'with the filter as it lies' not in got, got

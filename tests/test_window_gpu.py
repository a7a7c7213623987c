"""Convolutions over windows in LDS (csrc/winconv.hip): whole numbers, so that every result is compared value for value with numpy.
The sizes end tiles inside a row, between images and behind the last result, windows with one slab of channels, several of them
in one window or in two, and a last slab or block that is not full, columns anywhere; strides, dilations and paddings of any sign."""
import ctypes
import re

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
KINDS = {'f32': (hk.F32, hk.F32, lambda a: a, np.float32), 'bf16': (hk.BF16, hk.BF16, T.bf16, np.uint16),
         'i8': (hk.I8, hk.I32, lambda a: a.astype(np.int8), np.int32)}


@pytest.fixture(autouse=True)
def _device():
    hk.init(0)


def whole(rng, shape, top=3):
    return rng.integers(-top, top + 1, shape).astype(np.float32)


def run(kind, I, F, out_hw, stride, dil, pad, bias=None, relu=False, packed=True, tile=''):
    dt, out, cast, onp = KINDS[kind]
    d = hk.Conv2dDesc()
    d.in_dtype, d.out_dtype, d.c_dtype, d.flags = dt, out, out, hk.flag_conv(hk.CONV_WINDOW)
    d.n, d.h, d.w, d.ci = I.shape
    d.kh, d.kw, _, d.co = F.shape
    (d.oh, d.ow), (d.stride_h, d.stride_w), (d.dil_h, d.dil_w), (d.pad_h, d.pad_w) = out_hw, stride, dil, pad
    if relu:
        d.tail = hk.make_tail(ops=[(hk.EPI_RELU, out, 0, 0, 0.0)])
    if bias is not None:
        d.init_kind, d.init_dtype, d.init_row_stride, d.init_col_stride = 1, out, 0, 1
    L = hk.lib()
    plan = L.pml_hip_conv2d_dispatch(ctypes.byref(d))
    assert plan, L.pml_hip_last_error()
    assert 'over its window in LDS (' + tile in hk.describe(plan), hk.describe(plan)
    dI, dF = hk.DeviceBuffer.from_numpy(cast(I)), hk.DeviceBuffer.from_numpy(cast(F))
    dB = None if bias is None else hk.DeviceBuffer.from_numpy(cast(bias) if kind != 'i8' else bias.astype(np.int32))
    shape = (d.n, d.oh, d.ow, d.co)
    n = int(np.prod(shape))
    fill = np.full(n + 64, 77, onp)  # (what lies behind the result stays)
    dO, none = hk.DeviceBuffer.from_numpy(fill), hk.ptr_array([])
    if packed:
        hk.check(L.pml_hip_conv2d_pack_filter(plan, dF.ptr, None))
    for _ in range(2):
        hk.check(L.pml_hip_conv2d_invoke(plan, dI.ptr, None if packed else dF.ptr, dO.ptr, dB.ptr if dB else None, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(plan)
    got = dO.to_numpy(onp, (n + 64,))
    assert (got[n:] == 77).all()
    got = got[:n].reshape(shape)
    return E.bf16_from_bits(got) if kind == 'bf16' else got


def reference(I, F, out_hw, stride, dil, pad, bias=None, relu=False):
    (n, h, w, ci), (kh, kw, _, co), (oh, ow) = I.shape, F.shape, out_hw
    S = np.zeros((n, oh, ow, co), np.float64)
    for y in range(kh):
        for x in range(kw):
            ys, xs = np.arange(oh) * stride[0] + y * dil[0] - pad[0], np.arange(ow) * stride[1] + x * dil[1] - pad[1]
            yo, xo = (ys >= 0) & (ys < h), (xs >= 0) & (xs < w)
            if yo.any() and xo.any():
                part = I[:, ys[yo]][:, :, xs[xo]].astype(np.float32) @ F[y, x].astype(np.float32)  # (exact: sums below 2^24)
                S[np.ix_(np.arange(n), np.nonzero(yo)[0], np.nonzero(xo)[0])] += part
    if bias is not None:
        S += bias
    return np.maximum(S, 0) if relu else S


def compare(kind, got, want):
    np.testing.assert_array_equal(got, E.round_bf16(want.astype(np.float32)) if kind == 'bf16' else want)


# n, h, w, channels in 16-byte vectors, kh, kw, co, stride, dilation, padding (None: SAME)
SMALL = [
    (1, 3, 3, 4, 3, 3, 1, (1, 1), (1, 1), None),        # one tile, one column, images smaller than the filter's reach
    (5, 7, 7, 4, 3, 3, 33, (1, 1), (1, 1), None),       # tiles across images
    (3, 19, 17, 6, 3, 3, 40, (1, 1), (1, 1), None),     # a block and a half of channels, columns past the last whole eight
    (2, 23, 11, 8, 5, 3, 65, (1, 1), (1, 1), None),
    (2, 30, 31, 16, 7, 7, 23, (1, 1), (1, 1), None),    # several blocks in a window
    (2, 9, 40, 20, 1, 5, 100, (1, 1), (1, 2), None),    # filter rows only, five blocks of channels
    (4, 12, 13, 9, 2, 2, 70, (2, 2), (1, 1), None),     # windows side by side, two blocks and a quarter
    (3, 21, 20, 4, 3, 3, 31, (2, 3), (2, 1), None),
    (2, 15, 15, 32, 3, 3, 130, (2, 2), (1, 1), (0, 0)),  # windows past the image's end
    (2, 16, 18, 12, 3, 3, 64, (1, 1), (3, 2), (5, -2)),  # more padding than reach on one side, a cut on the other
    (6, 8, 8, 64, 3, 3, 48, (1, 1), (1, 1), None),      # 1 KB of channels
    (1, 1, 700, 4, 1, 3, 36, (1, 1), (1, 1), None),     # one row
    (1, 300, 1, 4, 3, 1, 36, (1, 1), (1, 1), None),     # one column
]


@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('case', SMALL, ids=lambda c: 'x'.join(map(str, c[:7])))
def test_small(kind, case):
    n, h, w, vectors, kh, kw, co, stride, dil, pad = case
    rng = np.random.default_rng(h * w + co)
    ci = vectors * {'f32': 4, 'bf16': 8, 'i8': 16}[kind]
    oh, ow = -(-h // stride[0]), -(-w // stride[1])
    if pad is None:
        pad = tuple(max(0, (o - 1) * s + (k - 1) * e + 1 - size) // 2 for o, s, k, e, size in zip((oh, ow), stride, (kh, kw), dil, (h, w)))
    I, F, bias = whole(rng, (n, h, w, ci)), whole(rng, (kh, kw, ci, co), 2), whole(rng, co, 50)
    geometry = ((oh, ow), stride, dil, pad)
    compare(kind, run(kind, I, F, *geometry, bias=bias, relu=True), reference(I, F, *geometry, bias=bias, relu=True))
    compare(kind, run(kind, I, F, *geometry, packed=False), reference(I, F, *geometry))


# sizes that take each configuration on a device of 256 compute units: many tiles, or few of them and a long K
LARGE = [('bf16', 128, 14, 256, 256, 3, 1, '8 wavefronts of 112x64, 2'), ('bf16', 101, 28, 128, 128, 3, 1, '4 wavefronts of 112x64)'),
         ('bf16', 127, 7, 512, 512, 3, 1, '8 wavefronts of 112x64, 4'), ('bf16', 40, 56, 128, 128, 3, 2, '8 wavefronts of 64x64, 2'),
         ('bf16', 16, 112, 64, 64, 3, 1, '4 wavefronts of 112x64)'), ('bf16', 15, 109, 32, 17, 3, 1, '4 wavefronts of 112x32)'),
         ('bf16', 84, 39, 32, 24, 3, 1, '4 wavefronts of 64x32)'), ('bf16', 64, 28, 64, 64, 3, 1, '4 wavefronts of 64x64, 2'),
         ('bf16', 79, 11, 128, 215, 3, 1, '8 wavefronts of 112x32, 2'), ('bf16', 3, 64, 128, 134, 5, 1, '4 wavefronts of 64x32, 2'),
         ('bf16', 39, 13, 128, 188, 7, 1, '4 wavefronts of 64x64, 4'), ('bf16', 18, 16, 64, 63, 5, 1, '8 wavefronts of 32x32, 4'),
         ('bf16', 95, 14, 256, 184, 5, 1, '8 wavefronts of 112x64, 4'), ('i8', 32, 56, 128, 64, 3, 1, '4 wavefronts of 112x64)'),
         ('i8', 7, 114, 128, 134, 3, 1, '4 wavefronts of 64x32)'), ('f32', 16, 56, 64, 64, 3, 1, '8 wavefronts of 112x64, 4'),
         ('f32', 17, 45, 64, 215, 3, 1, '4 wavefronts of 64x32)')]


@pytest.mark.parametrize('kind,n,hw,ci,co,k,s,tile', LARGE)
def test_large(kind, n, hw, ci, co, k, s, tile):
    rng = np.random.default_rng(hw)
    I, F, bias = whole(rng, (n, hw, hw, ci), 2), whole(rng, (k, k, ci, co), 1), whole(rng, co, 50)
    o = -(-hw // s)
    p = max(0, (o - 1) * s + k - hw) // 2
    geometry = ((o, o), (s, s), (1, 1), (p, p))
    compare(kind, run(kind, I, F, *geometry, bias=bias, relu=True, packed=co % 2 == 0, tile=tile), reference(I, F, *geometry, bias=bias, relu=True))


@pytest.mark.parametrize('kind', ['f32', 'bf16'])
def test_infinities_stay_with_their_taps(kind):
    """Channels that end inside a block: what stands beside a pixel's last channels and a tap's last weights is no term."""
    rng = np.random.default_rng(5)
    ci = {'f32': 4, 'bf16': 8}[kind] * 6
    I, F = np.abs(whole(rng, (2, 12, 12, ci))) + 1, np.abs(whole(rng, (3, 3, ci, 20), 2)) + 1
    geometry = ((10, 10), (1, 1), (1, 1), (0, 0))
    want = reference(I, F, *geometry)
    Fi, Ii = F.copy(), I.copy()
    Fi[1, 1, 0, 3] = np.inf
    Ii[1, 4, 5, 0] = np.nan
    got = run(kind, Ii, Fi, *geometry)
    touched = np.zeros(want.shape, bool)
    touched[1, 2:5, 3:6] = True
    want[..., 3] = np.inf
    assert np.isnan(got[touched]).all()
    compare(kind, got[~touched], want[~touched])



# every configuration of every type, on a device of 256 compute units: n, height and width, channels, columns, filter, stride; the
# columns of a tile, its wavefronts, what each of them holds, how many share K
EVERY = [('bf16', 75, 53, 64, 20, 2, 1, 32, 4, '112x32', 1), ('bf16', 3, 56, 32, 125, 2, 1, 32, 4, '64x32', 1),
         ('bf16', 10, 53, 32, 17, 2, 1, 32, 4, '64x32', 2), ('bf16', 1, 8, 64, 30, 2, 2, 32, 8, '32x32', 4),
         ('bf16', 41, 45, 32, 33, 2, 1, 64, 4, '112x64', 1), ('bf16', 49, 21, 32, 189, 3, 2, 64, 4, '64x64', 2),
         ('bf16', 77, 25, 128, 78, 2, 2, 64, 4, '64x64', 4), ('bf16', 10, 60, 256, 54, 2, 1, 64, 8, '112x64', 4),
         ('bf16', 68, 47, 32, 56, 2, 2, 128, 4, '112x64', 1), ('bf16', 90, 30, 32, 72, 2, 2, 128, 8, '112x32', 2),
         ('bf16', 18, 55, 128, 289, 2, 2, 128, 8, '112x64', 2), ('bf16', 66, 17, 128, 74, 5, 1, 128, 8, '112x64', 4),
         ('bf16', 14, 54, 64, 299, 2, 2, 128, 8, '64x64', 2), ('f32', 33, 57, 16, 20, 2, 1, 32, 4, '112x32', 1),
         ('f32', 11, 63, 16, 19, 3, 1, 32, 4, '64x32', 1), ('f32', 16, 41, 16, 22, 2, 1, 32, 4, '64x32', 2),
         ('f32', 3, 19, 16, 51, 2, 1, 32, 8, '32x32', 4), ('f32', 22, 45, 32, 287, 3, 1, 64, 4, '112x64', 1),
         ('f32', 36, 50, 32, 39, 3, 1, 64, 4, '64x64', 2), ('f32', 98, 17, 64, 54, 5, 1, 64, 4, '64x64', 4),
         ('f32', 81, 26, 64, 43, 3, 1, 64, 8, '112x64', 4), ('f32', 82, 36, 64, 114, 2, 1, 128, 4, '112x64', 1),
         ('f32', 4, 56, 32, 196, 3, 1, 128, 8, '112x32', 2), ('f32', 44, 24, 64, 249, 3, 1, 128, 8, '112x64', 2),
         ('f32', 42, 19, 64, 197, 2, 1, 128, 8, '64x64', 2), ('i8', 45, 63, 64, 17, 3, 1, 32, 4, '112x32', 1),
         ('i8', 11, 61, 64, 25, 2, 1, 32, 4, '64x32', 1), ('i8', 34, 34, 64, 87, 2, 2, 32, 4, '64x32', 2),
         ('i8', 1, 6, 64, 18, 2, 1, 32, 8, '32x32', 4), ('i8', 44, 51, 64, 44, 2, 1, 64, 4, '112x64', 1),
         ('i8', 7, 60, 64, 190, 2, 2, 64, 4, '64x64', 2), ('i8', 98, 19, 512, 34, 2, 2, 64, 4, '64x64', 4),
         ('i8', 11, 54, 512, 21, 3, 1, 64, 8, '112x64', 4), ('i8', 14, 51, 64, 40, 2, 1, 128, 4, '112x64', 1),
         ('i8', 65, 16, 64, 49, 2, 1, 128, 8, '112x32', 2), ('i8', 18, 46, 64, 66, 5, 1, 128, 8, '112x64', 2),
         ('i8', 15, 45, 128, 34, 3, 1, 128, 8, '64x64', 2)]


@pytest.mark.parametrize('kind,n,hw,ci,co,k,s,columns,wavefronts,block,sharing', EVERY)
def test_every_configuration(kind, n, hw, ci, co, k, s, columns, wavefronts, block, sharing):
    o = -(-hw // s)
    p = max(0, (o - 1) * s + k - hw) // 2
    d = hk.Conv2dDesc()
    d.in_dtype, (d.out_dtype, d.c_dtype) = KINDS[kind][0], [KINDS[kind][1]] * 2
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, hw, hw, ci, k, k, co, o, o
    d.stride_h, d.stride_w, d.dil_h, d.dil_w, d.pad_h, d.pad_w = s, s, 1, 1, p, p
    plan = hk.lib().pml_hip_conv2d_dispatch(ctypes.byref(d))
    text = hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    shared = ', %d sharing K' % sharing if sharing > 1 else ''
    assert re.search(r'tile=\d+x%d over its window in LDS \(%d wavefronts of %s%s\)' % (columns, wavefronts, block, shared), text), text
    rng = np.random.default_rng(hw + co)
    I, F, bias = whole(rng, (n, hw, hw, ci), 2), whole(rng, (k, k, ci, co), 1), whole(rng, co, 50)
    geometry = ((o, o), (s, s), (1, 1), (p, p))
    compare(kind, run(kind, I, F, *geometry, bias=bias, relu=True, tile='%d wavefronts of %s%s)' % (wavefronts, block, shared)), reference(I, F, *geometry, bias=bias, relu=True))


# 64-byte blocks of channels fewer than the wavefronts that share K, as many, and more; filter rows of fewer taps than a step counts on
@pytest.mark.parametrize('kind', ['f32', 'bf16', 'i8'])
@pytest.mark.parametrize('vectors,kh,kw', [(4, 2, 2), (4, 7, 1), (4, 1, 7), (8, 3, 1), (8, 2, 3), (12, 1, 4), (12, 7, 2), (16, 4, 1), (16, 1, 5), (16, 5, 5), (20, 2, 1), (28, 3, 2), (36, 1, 3)])
def test_steps_counted_over_blocks_and_taps(kind, vectors, kh, kw):
    rng = np.random.default_rng(vectors * 100 + kh * 10 + kw)
    ci, n, h, w, co = vectors * {'f32': 4, 'bf16': 8, 'i8': 16}[kind], 2, 9, 8, 20
    pad = ((kh - 1) // 2, (kw - 1) // 2)
    I, F = whole(rng, (n, h, w, ci)), whole(rng, (kh, kw, ci, co), 2)
    geometry = ((h, w), (1, 1), (1, 1), pad)
    compare(kind, run(kind, I, F, *geometry), reference(I, F, *geometry))

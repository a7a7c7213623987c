"""A convolution's gradients at the edges of their kernels: runs cut by the image, the filter row and the tensor's end; splits of the
pixels; columns of channel counts that are no multiple of a vector; padded gradients."""
import ctypes

import numpy as np
import pytest
import torch

from plaidml_amd import edsl as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


def gradients(x, f, g, stride, pad, dil):
    """Both gradients in 64 bits (NHWC, HWCK)."""
    n, h, w, ci = x.shape
    kh, kw, _, co = f.shape
    oh, ow = g.shape[1:3]
    X = torch.from_numpy(x).double().permute(0, 3, 1, 2).requires_grad_()
    F = torch.from_numpy(f).double().permute(3, 2, 0, 1).requires_grad_()
    below = (oh - 1) * stride + (kh - 1) * dil + 1 - h - pad
    right = (ow - 1) * stride + (kw - 1) * dil + 1 - w - pad
    y = torch.nn.functional.conv2d(torch.nn.functional.pad(X, (pad, right, pad, below)), F, stride=stride, dilation=dil)
    assert tuple(y.shape) == (n, co, oh, ow)
    y.backward(torch.from_numpy(g).double().permute(0, 3, 1, 2))
    return X.grad.permute(0, 2, 3, 1).numpy(), F.grad.permute(2, 3, 1, 0).numpy()


CASES = [  # n, h, w, ci, kh, kw, co, oh, ow, stride, pad, dil
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 1),         # tensors shorter than one load
    (1, 2, 1, 3, 3, 3, 2, 2, 1, 1, 1, 1),         # every window cut on both sides
    (2, 5, 7, 3, 3, 3, 5, 5, 7, 1, 1, 1),
    (1, 9, 9, 15, 5, 5, 20, 9, 9, 1, 2, 1),
    (3, 11, 6, 22, 3, 3, 67, 11, 6, 1, 1, 1),     # window rows of 66 values, columns of 67: one tile and a rest of both
    (2, 13, 9, 5, 3, 3, 9, 7, 5, 2, 1, 1),        # columns: channel chunks that overlap
    (1, 12, 12, 7, 5, 5, 33, 4, 4, 3, 1, 1),
    (2, 8, 8, 3, 1, 1, 4, 4, 4, 2, 0, 1),         # pixels that no window covers
    (1, 15, 1, 6, 3, 1, 8, 7, 1, 2, 0, 2),        # rows of taps apart
    (5, 40, 41, 6, 3, 3, 18, 40, 41, 1, 1, 1),    # 128 slabs and a piece: splits of two slabs
    (9, 64, 64, 17, 3, 3, 38, 64, 64, 1, 1, 1),   # splits that several threads add up
]


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('case', CASES, ids=lambda c: 'x'.join(map(str, c)))
def test_gradients(case, dtype):
    n, h, w, ci, kh, kw, co, oh, ow, stride, pad, dil = case
    print(case, dtype, flush=True)
    hk.init(0)
    L = hk.lib()
    rng = np.random.default_rng(sum(case))
    bf = dtype == 'bf16'
    x, f, g = (E.round_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((n, h, w, ci), (kh, kw, ci, co), (n, oh, ow, co)))
    want_x, want_f = gradients(x, f, g, stride, pad, dil)
    d = hk.Conv2dDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16 if bf else hk.F32
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, w, ci, kh, kw, co, oh, ow
    d.stride_h = d.stride_w = stride
    d.pad_h = d.pad_w = pad
    d.dil_h = d.dil_w = dil
    dev = [hk.DeviceBuffer.from_numpy(E.to_bf16_bits(a) if bf else a) for a in (x, f, g)]
    L.pml_hip_conv2d_grad_dispatch.restype = ctypes.c_int64
    for which, other, want in ((0, dev[1], want_x), (1, dev[0], want_f)):
        if not L.pml_hip_conv2d_grad_takes(ctypes.byref(d), which):
            continue
        p = L.pml_hip_conv2d_grad_dispatch(ctypes.byref(d), which)
        assert p, L.pml_hip_last_error()
        terms = kh * kw * co if which == 0 else n * oh * ow
        out = hk.DeviceBuffer.from_numpy(np.full(want.size, np.nan, np.float32).astype(np.float32))
        for _ in range(2):
            hk.check(L.pml_hip_conv2d_grad_invoke(ctypes.c_int64(p), ctypes.c_void_p(dev[2].ptr), ctypes.c_void_p(other.ptr), ctypes.c_void_p(out.ptr), None))
        hk.check(L.pml_hip_stream_sync(None))
        got = E.from_bf16_bits(out.to_numpy(np.uint16, want.shape)) if bf else out.to_numpy(np.float32, want.shape)
        # products of bf16 values are exact in fp32; a sum of t terms of size one is off by sqrt(t) roundings of a partial sum of
        # size sqrt(t), 2^-24 of it each, and where the result is bf16 by 2^-9 of itself
        bound = 4 * terms * 2.0 ** -24 + (2.0 ** -8 * np.abs(want) if bf else 4 * 2.0 ** -24)
        np.testing.assert_array_less(np.abs(got.astype(np.float64) - want), bound + 1e-30)
        hk.lib().pml_hip_plan_free(ctypes.c_int64(p))


MORE = [
    (3, 9, 7, 13, 1, 1, 20, 3, 2, 3, 0, 1),       # one tap: pixels that no window covers, pixels behind the last gradient row and column
    (1, 11, 10, 5, 1, 1, 9, 6, 6, 2, 1, 1),       # ... and gradient pixels beside the image
    (2, 21, 11, 150, 3, 3, 80, 21, 11, 1, 1, 1),  # 300 KB of results a split
    (1, 46, 45, 90, 5, 5, 9, 46, 45, 1, 2, 1),    # many pixels of long windows, bf16: run by run again
    (2, 8, 8, 10, 3, 3, 6, 8, 8, 1, 1, 1),        # two slabs of bf16 pixels, and more
    (2, 9, 8, 10, 3, 3, 6, 9, 8, 1, 1, 1),
]


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('case', MORE, ids=lambda c: 'x'.join(map(str, c)))
def test_gradients_of_one_tap_and_of_few_splits(case, dtype):
    test_gradients(case, dtype)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('case', CASES + MORE, ids=lambda c: 'x'.join(map(str, c)))
def test_every_case_is_taken(case, dtype):
    """Both gradients of every case above, by columns or with the splits that it is there for."""
    n, h, w, ci, kh, kw, co, oh, ow, stride, pad, dil = case
    L = hk.lib()
    d = hk.Conv2dDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16 if dtype == 'bf16' else hk.F32
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, w, ci, kh, kw, co, oh, ow
    d.stride_h = d.stride_w = stride
    d.pad_h = d.pad_w = pad
    d.dil_h = d.dil_w = dil
    L.pml_hip_conv2d_grad_dispatch.restype = ctypes.c_int64
    for which in (0, 1):
        assert L.pml_hip_conv2d_grad_takes(ctypes.byref(d), which) == 1
        p = L.pml_hip_conv2d_grad_dispatch(ctypes.byref(d), which)
        assert p, L.pml_hip_last_error()
        text = hk.describe(ctypes.c_int64(p))
        L.pml_hip_plan_free(ctypes.c_int64(p))
        if which == 0:
            assert ('as a convolution of the gradient' if stride == 1 else 'by columns') in text, text
            assert 'as it lies' not in text, text  # (the flipped filter is laid out by every call)
        else:  # (pixels over one workgroup, over splits of two slabs, over more than a thread adds up)
            splits = int(text.split('splits=')[1].split()[0])
            assert splits >= (9 if n * oh * ow > 30000 else 2 if n * oh * ow > 1000 else 1), text


# one tap, where the stride is one in one direction; several
@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('stride,k', [((1, 2), 1), ((2, 1), 1), ((3, 2), 1), ((1, 2), 2), ((1, 1), 1)])
def test_gradients_of_a_cropped_image(stride, k, dtype):
    """A negative padding crops: pixels ahead of the first window take no gradient, and no filter gradient takes them."""
    n, h, w, ci, co, crop = 2, 9, 12, 6, 5, (2, 1)
    oh, ow = (h - crop[0] - k) // stride[0], (w - crop[1] - k) // stride[1]
    print(stride, k, dtype, flush=True)
    hk.init(0)
    L, rng, bf = hk.lib(), np.random.default_rng(k), dtype == 'bf16'
    x, f, g = (E.round_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((n, h, w, ci), (k, k, ci, co), (n, oh, ow, co)))
    want_x, want_f = np.zeros((n, h, w, ci)), np.zeros((k, k, ci, co))
    for ky in range(k):
        for kx in range(k):
            at = (slice(None), slice(crop[0] + ky, crop[0] + ky + oh * stride[0], stride[0]), slice(crop[1] + kx, crop[1] + kx + ow * stride[1], stride[1]))
            want_x[at] += g.astype(np.float64) @ f[ky, kx].T
            want_f[ky, kx] = np.tensordot(x[at].astype(np.float64), g, ((0, 1, 2), (0, 1, 2)))
    d = hk.Conv2dDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.BF16 if bf else hk.F32
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, h, w, ci, k, k, co, oh, ow
    d.stride_h, d.stride_w = stride
    d.pad_h, d.pad_w = -crop[0], -crop[1]
    d.dil_h = d.dil_w = 1
    dev = [hk.DeviceBuffer.from_numpy(E.to_bf16_bits(a) if bf else a) for a in (x, f, g)]
    L.pml_hip_conv2d_grad_dispatch.restype = ctypes.c_int64
    for which, other, want in ((0, dev[1], want_x), (1, dev[0], want_f)):
        assert L.pml_hip_conv2d_grad_takes(ctypes.byref(d), which) == 1
        p = L.pml_hip_conv2d_grad_dispatch(ctypes.byref(d), which)
        assert p, L.pml_hip_last_error()
        out = hk.DeviceBuffer.from_numpy(np.full(want.size, np.nan, np.float32))
        hk.check(L.pml_hip_conv2d_grad_invoke(ctypes.c_int64(p), ctypes.c_void_p(dev[2].ptr), ctypes.c_void_p(other.ptr), ctypes.c_void_p(out.ptr), None))
        got = E.from_bf16_bits(out.to_numpy(np.uint16, want.shape)) if bf else out.to_numpy(np.float32, want.shape)
        L.pml_hip_plan_free(ctypes.c_int64(p))
        terms = k * k * co if which == 0 else n * oh * ow
        np.testing.assert_allclose(got, want, rtol=2.0 ** -8 if bf else 2.0 ** -20, atol=terms * 2.0 ** -22)

"""Products over free strides and the gradients of a convolution (csrc/strided.hip) against float64 on the CPU, at the sizes where
tiles, slabs, splits and 16-byte vectors end raggedly."""
import ctypes

import numpy as np
import pytest
import torch

from plaidml_amd import edsl as P
from plaidml_amd import hipkernels as hk
from plaidml_amd import op as Pop

pytestmark = pytest.mark.gpu
DT = {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16}


def values(rng, shape, dtype, scale=1.0):
    a = rng.standard_normal(shape).astype(np.float32) * np.float32(scale)
    return P.round_bf16(a) if dtype == 'bf16' else a


def check(got, want, dtype):
    err = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
    assert np.isfinite(got).all() and err < (6e-3 if dtype == 'bf16' else 2e-6), err


def plan_of(program):
    return [v for k, v in program.passes if k == 'hip-plan'][0]


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('b,m,n,k,ta,tb', [
    (1, 1, 1, 2, 0, 0), (1, 300, 777, 1001, 0, 0), (3, 64, 64, 64, 0, 1), (5, 65, 31, 33, 0, 0), (2, 127, 129, 100, 1, 0),
    (7, 19, 276, 32, 0, 1), (1, 130, 70, 5003, 1, 0), (2, 3, 5, 7, 1, 1), (1, 1100, 2051, 67, 0, 0), (4, 1, 33, 130, 0, 1),
    (300, 100, 100, 40, 1, 0), (300, 128, 65, 70, 0, 1), (300, 64, 70, 33, 1, 1)])  # (many tiles: of 128, and of 64 where those would be empty)
def test_product(dtype, b, m, n, k, ta, tb):
    rng = np.random.default_rng(m * 7 + n)
    A, B = values(rng, (b, k, m) if ta else (b, m, k), dtype), values(rng, (b, n, k) if tb else (b, k, n), dtype, k ** -0.5)
    bias = values(rng, (n,), dtype)
    X, Y, Z = (P.Placeholder(DT[dtype], x.shape) for x in (A, B, bias))
    bi, i, j, q = P.TensorIndexes(4)
    C = P.Contraction().outShape(b, m, n).outAccess(bi, i, j).sum((X[bi, q, i] if ta else X[bi, i, q]) * (Y[bi, j, q] if tb else Y[bi, q, j])).build()
    program = P.Program('product', [X, Y, Z], [Pop.relu(C * 0.5 + Z)])
    got, = P.Runner(program, target='hip').run([A, B, bias])
    want = np.matmul((A.transpose(0, 2, 1) if ta else A).astype(np.float64), (B.transpose(0, 2, 1) if tb else B).astype(np.float64))
    check(got, np.maximum(want * 0.5 + bias, 0), dtype)
    assert 'general' not in plan_of(program)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('tb', [0, 1])
@pytest.mark.parametrize('b,m,n,k', [
    (1, 1, 4, 1), (1, 3, 66, 31), (1, 16, 61, 33), (2, 17, 67, 96), (1, 33, 131, 255), (3, 32, 65, 257), (1, 31, 5, 300), (9, 100, 77, 100)])
def test_product_of_few_tiles(dtype, tb, b, m, n, k):
    """Direct tiles of 16 or 32 rows by 64 columns: one, two and three columns past a quad, K short of a step, of whole steps
    only, and with one value left; an infinity in the last row and column of B stays in its own results."""
    rng = np.random.default_rng(m + n + k)
    A, B = values(rng, (b, m, k), dtype), values(rng, (b, n, k) if tb else (b, k, n), dtype, k ** -0.5)
    A = np.abs(A) + 1
    (B[:, n - 1:, k - 1] if tb else B[:, k - 1, n - 1:])[...] = np.inf
    X, Y = P.Placeholder(DT[dtype], A.shape), P.Placeholder(DT[dtype], B.shape)
    bi, i, j, q = P.TensorIndexes(4)
    C = P.Contraction().outShape(b, m, n).outAccess(bi, i, j).sum(X[bi, i, q] * (Y[bi, j, q] if tb else Y[bi, q, j])).build()
    got, = P.Runner(P.Program('product', [X, Y], [C]), target='hip').run([P.round_bf16(A) if dtype == 'bf16' else A, B])
    A = (P.round_bf16(A) if dtype == 'bf16' else A).astype(np.float64)
    want = np.matmul(A, (B.transpose(0, 2, 1) if tb else B).astype(np.float64))
    assert np.isposinf(got[..., -1]).all()
    check(got[..., :-1], want[..., :-1], dtype)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('n,hw,ci,co,k,stride', [
    (2, 14, 64, 64, 3, 1), (1, 7, 3, 16, 3, 2), (3, 9, 19, 33, 5, 1), (2, 15, 70, 20, 3, 2), (1, 10, 5, 17, 1, 2), (2, 8, 24, 40, 1, 1),
    (1, 112, 3, 37, 5, 1), (5, 11, 130, 65, 3, 1), (1, 2, 8, 16, 3, 1), (4, 40, 16, 24, 5, 2)])
def test_conv_gradients(dtype, n, hw, ci, co, k, stride):
    rng = np.random.default_rng(hw * 3 + co)
    o = (hw + stride - 1) // stride
    Iv, Fv, Gv = values(rng, (n, hw, hw, ci), dtype), values(rng, (k, k, ci, co), dtype, (k * k * co) ** -0.5), values(rng, (n, o, o, co), dtype)
    X, F, G = (P.Placeholder(DT[dtype], x.shape) for x in (Iv, Fv, Gv))
    dX = Pop.convolution(G, F, strides=[stride, stride], deriv_mode=Pop.DERIV_DATA, result_shape=[hw, hw])
    dF = Pop.convolution(X, G, strides=[stride, stride], deriv_mode=Pop.DERIV_FILTER, result_shape=[k, k])
    program = P.Program('gradients', [X, F, G], [dX, dF])
    runner = P.Runner(program, target='hip')
    for _ in range(4):  # one by one, then as a recorded graph
        gx, gf = runner.run([Iv, Fv, Gv])
    before = max(0, (o - 1) * stride + k - hw) // 2
    x = torch.nn.functional.pad(torch.from_numpy(Iv).double().permute(0, 3, 1, 2), (before, k + stride, before, k + stride)).requires_grad_(True)
    f = torch.from_numpy(Fv).double().permute(3, 2, 0, 1).requires_grad_(True)
    y = torch.nn.functional.conv2d(x, f, stride=stride)[:, :, :o, :o]
    y.backward(torch.from_numpy(Gv).double().permute(0, 3, 1, 2))
    check(gx, x.grad[:, :, before:before + hw, before:before + hw].permute(0, 2, 3, 1).numpy(), dtype)
    check(gf, f.grad.permute(2, 3, 1, 0).numpy(), dtype)
    assert 'general' not in plan_of(program)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('n,h,w,ci,co,k,stride', [
    (2, 14, 14, 64, 64, 3, 1), (16, 56, 56, 64, 64, 3, 1), (1, 7, 9, 3, 16, 3, 2), (3, 9, 8, 19, 33, 5, 1), (2, 12, 15, 70, 20, 3, 2),
    (1, 5, 6, 64, 96, 1, 1), (2, 3, 2, 8, 24, 5, 1)])
def test_conv_gradients_leave_taps_outside_out(dtype, n, h, w, ci, co, k, stride):
    """Taps that leave the image are no terms of either gradient: an infinity or a NaN in the gradient's border (filter
    gradient) or in the filter (data gradient) is in the results that it reaches and in no other.  Sums of up to a tile, of
    split K, of every convolution kernel the data gradient runs on, image rows of their own length."""
    rng = np.random.default_rng(h * 3 + co)
    oh, ow = (h + stride - 1) // stride, (w + stride - 1) // stride
    py, px = (max(0, (o - 1) * stride + k - s) // 2 for o, s in ((oh, h), (ow, w)))
    Iv, Fv, Gv = values(rng, (n, h, w, ci), dtype), values(rng, (k, k, ci, co), dtype, (k * k * co) ** -0.5), values(rng, (n, oh, ow, co), dtype)
    # (one of a kind per channel: a sum holds one infinity, whose sign is known, or a NaN of its own)
    Gv[0, 0, 0, 0], Gv[n - 1, oh - 1, ow // 2, 1], Gv[0, oh // 2, ow - 1, 2] = np.inf, np.nan, -np.inf
    Gv[n - 1, 0, :, co - 1] = np.inf
    Fv[0, 0, 0, 3], Fv[k - 1, 0, ci - 1, 4], Fv[k // 2, k - 1, 1, 5] = np.inf, np.nan, -np.inf
    finite_f, finite_g = np.where(np.isfinite(Fv), Fv, 0.5).astype(np.float32), np.where(np.isfinite(Gv), Gv, 0.5).astype(np.float32)
    X, F, G = (P.Placeholder(DT[dtype], x.shape) for x in (Iv, Fv, Gv))
    dX = Pop.convolution(G, F, strides=[stride, stride], deriv_mode=Pop.DERIV_DATA, result_shape=[h, w])
    dF = Pop.convolution(X, G, strides=[stride, stride], deriv_mode=Pop.DERIV_FILTER, result_shape=[k, k])
    runner = P.Runner(P.Program('gradients', [X, F, G], [dX, dF]), target='hip')
    gf = runner.run([Iv, finite_f, Gv])[1]
    gx = runner.run([Iv, Fv, finite_g])[0]
    want_x, want_f = np.zeros((n, h, w, ci)), np.zeros((k, k, ci, co))
    with np.errstate(invalid='ignore'):
        for ky in range(k):
            for kx in range(k):
                ys = [y for y in range(oh) if 0 <= y * stride + ky - py < h]
                xs = [x for x in range(ow) if 0 <= x * stride + kx - px < w]
                if not ys or not xs:
                    continue
                at = np.ix_(range(n), [y * stride + ky - py for y in ys], [x * stride + kx - px for x in xs])
                of = np.ix_(range(n), ys, xs)
                for c in range(ci):  # (term by term: a zero weight of a matrix product would itself make NaNs)
                    want_x[at + (c,)] += (finite_g[of].astype(np.float64) * Fv[ky, kx, c]).sum(-1)
                    want_f[ky, kx, c] = (Iv[at + (c,)].astype(np.float64)[..., None] * Gv[of]).sum((0, 1, 2))
    assert not np.isfinite(want_f).all() and (k > w or not np.isfinite(want_x).all())  # (5 taps over 2 pixels: those three are never inside)
    for got, want in ((gx, want_x), (gf, want_f)):
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
        np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
        check(got[np.isfinite(want)], want[np.isfinite(want)], dtype)


@pytest.mark.parametrize('nk', [0, 1])
@pytest.mark.parametrize('at', [0, 1])
@pytest.mark.parametrize('b,m,n,k', [(1, 1, 4, 65), (1, 3, 2050, 95), (2, 17, 67, 33), (1, 33, 65, 257), (1, 16, 64, 512), (3, 15, 66, 66), (1, 40, 5, 1001), (260, 33, 7, 31), (9, 31, 70, 287)])
def test_bf16_rows_that_begin_off_a_word(nk, at, b, m, n, k):
    """Direct bf16 tiles over matrices that begin at an odd value or not, with rows a few values longer than K or N and NaN in
    all that belongs to neither matrix: whole and broken steps of K, one and two rounds of steps, columns past a quad."""
    rng = np.random.default_rng(m * n + k + at)
    pa, pb, pc = k + 3 - at, (k if nk else n) + 2 + at, n + 1
    rows_b = n if nk else k

    def embed(rows, cols, pitch):
        v = P.round_bf16(rng.standard_normal((b, rows, cols)).astype(np.float32))
        flat = torch.full((at + b * rows * pitch + 4,), float('nan'), dtype=torch.bfloat16, device='cuda')
        flat[at:at + b * rows * pitch].view(b, rows, pitch)[:, :, :cols] = torch.from_numpy(v).to('cuda', torch.bfloat16)
        return v.astype(np.float64), flat
    A, da = embed(m, k, pa)
    B, db = embed(rows_b, k if nk else n, pb)
    out = torch.full((at + b * m * pc + 4,), 7.0, dtype=torch.bfloat16, device='cuda')
    d = hk.ProductDesc()
    d.in_dtype = d.out_dtype = hk.BF16
    d.n_batch, d.m, d.n, d.k, d.a_ms, d.a_ks, d.c_ms, d.row_len = 1, m, n, k, pa, 1, pc, n
    d.batch[0], d.a_batch[0], d.b_batch[0], d.c_batch[0] = b, m * pa, rows_b * pb, m * pc
    d.b_ks, d.b_ns = (1, pb) if nk else (pb, 1)
    L = hk.lib()
    plan = L.pml_hip_product_dispatch(ctypes.byref(d))
    text = hk.describe(plan)
    assert 'tile=16x64' in text or 'tile=32x64' in text, text
    torch.cuda.synchronize()
    hk.check(L.pml_hip_product_invoke(plan, da.data_ptr() + 2 * at, db.data_ptr() + 2 * at, out.data_ptr() + 2 * at, None, None, None))
    torch.cuda.synchronize()
    L.pml_hip_plan_free(plan)
    got = out[at:at + b * m * pc].view(b, m, pc).float().cpu().numpy()
    assert (got[:, :, n:] == 7).all() and (out[at + b * m * pc:] == 7).all() and (out[:at] == 7).all()
    want = np.matmul(A, B.transpose(0, 2, 1) if nk else B)
    # rounding to bf16 (2^-9), and fp32 sums of k products whichever way they are ordered
    bound = np.abs(want) * 2.0 ** -8 + np.matmul(np.abs(A), np.abs(B.transpose(0, 2, 1) if nk else B)) * (k * 2.0 ** -23)
    assert (np.abs(got[:, :, :n] - want) <= bound).all()

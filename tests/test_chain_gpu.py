"""Two products in a row as one launch (csrc/chain.hip): whole numbers, so that both results are compared value for value with
numpy; rows that end inside a step, rows of operands longer than they are wide, every width that is built."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from oracle import tile_oplib as Eop
from plaidml_amd import edsl as P
from plaidml_amd import hipkernels as hk
from plaidml_amd import op as Pop


def descs(m, k, k2, n, n2, residual, gap=0, relu=True):
    def one(rows, cols, terms, res):
        g = hk.GemmDesc()
        g.in_dtype = g.out_dtype = g.c_dtype = hk.BF16
        g.m, g.n, g.k, g.lda, g.ldb, g.ldc = rows, cols, terms, terms + gap, cols, cols + gap
        g.init_kind, g.init_dtype, g.init_row_stride, g.init_col_stride = 1, hk.BF16, 0, 1
        ops = ([(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0)] if res else []) + ([(hk.EPI_RELU, hk.BF16, 0, 0, 0.0)] if relu else [])
        g.tail = hk.make_tail(ops=ops, operands=[(hk.BF16, cols + gap, 1)] if res else [])
        return g
    first, second = one(m, n, k, residual), one(m, n2, n, False)
    if k2:
        first.k2, first.lda2, first.ldb2, first.init2_kind = k2, k2 + gap, n, 1
    return first, second


WIDTHS = [(64, 0, 256, 64), (64, 0, 256, 128), (128, 0, 256, 64), (32, 32, 256, 64), (64, 64, 256, 64), (96, 32, 256, 64), (128, 0, 512, 128), (96, 32, 512, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize('k,k2,n,n2', WIDTHS)
@pytest.mark.parametrize('m,gap,residual,relu', [(4096, 0, True, True), (4097, 8, False, True), (12295, 16, True, False), (16384 + 15, 0, False, False)])
def test_both_results(k, k2, n, n2, m, gap, residual, relu):
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    if k2 and residual:
        residual = False  # (a residual and a second part are not one launch: test_what_is_taken)
    rng = np.random.default_rng(m + n2 + k)

    def whole(rows, cols, top=2):
        return rng.integers(-top, top + 1, (rows, cols)).astype(np.float32)
    A, A2, R = whole(m, k + gap), whole(m, max(k2, 1) + gap), whole(m, n + gap, 30)
    B, B2, Bn = whole(k, n, 1), whole(max(k2, 1), n, 1), whole(n, n2, 1)
    b, b2, bn = whole(1, n, 9)[0], whole(1, n, 9)[0], whole(1, n2, 9)[0]
    A[5, 3], A[m - 1, 0] = np.nan, np.inf
    first, second = descs(m, k, k2, n, n2, residual, gap, relu)
    assert L.pml_hip_gemm_chain_takes(ctypes.byref(first), ctypes.byref(second))
    plans = [L.pml_hip_gemm_dispatch(ctypes.byref(d)) for d in (first, second)]
    dA, dA2, dR, dB, dB2, dBn, db, db2, dbn = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, A2, R, B, B2, Bn, b, b2, bn))
    dC, dD = (hk.DeviceBuffer.from_numpy(np.full((m + 1) * (c + gap), 77, np.uint16)) for c in (n, n2))
    hk.check(L.pml_hip_gemm_pack_b(plans[0], dB.ptr, None))
    hk.check(L.pml_hip_gemm_pack_b(plans[1], dBn.ptr, None))
    if k2:
        hk.check(L.pml_hip_gemm_pack_b2(plans[0], dB2.ptr, None))
    for _ in range(2):
        hk.check(L.pml_hip_gemm_chain_invoke(plans[0], plans[1], dA.ptr, dC.ptr, db.ptr, dA2.ptr if k2 else None, db2.ptr,
                                             hk.ptr_array([dR.ptr]) if residual else none, dD.ptr, dbn.ptr, None))
    hk.check(L.pml_hip_stream_sync(None))
    for p in plans:
        L.pml_hip_plan_free(p)
    C, D = dC.to_numpy(np.uint16, (m + 1, n + gap)), dD.to_numpy(np.uint16, (m + 1, n2 + gap))
    assert (C[m] == 77).all() and (D[m] == 77).all() and (C[:m, n:] == 77).all() and (D[:m, n2:] == 77).all()
    with np.errstate(invalid='ignore'):
        want = A[:, :k] @ B + b + (A2[:, :k2] @ B2 + b2 if k2 else 0)
        want = E.round_bf16(E.round_bf16(want.astype(np.float32)) + R[:, :n]) if residual else E.round_bf16(want.astype(np.float32))
        if relu:
            want = np.where(want < 0, 0, want)
        got = E.bf16_from_bits(C[:m, :n])
        np.testing.assert_array_equal(got, want)
        then = E.round_bf16((want @ Bn + bn).astype(np.float32))  # (exact: whole numbers below 2^24)
        if relu:
            then = np.where(then < 0, 0, then)
    np.testing.assert_array_equal(E.bf16_from_bits(D[:m, :n2]), then)


def test_what_is_taken():
    """Descriptors only: no device is asked."""
    def takes(*args, change=None, **kw):
        first, second = descs(*args, **kw)
        if change:
            change(first, second)
        return bool(hk.lib().pml_hip_gemm_chain_takes(ctypes.byref(first), ctypes.byref(second)))
    for k, k2, n, n2 in WIDTHS:
        assert takes(8192, k, k2, n, n2, False) and takes(8192, k, k2, n, n2, True) == (k2 == 0)
        assert not takes(16, k, k2, n, n2, False)
    assert not takes(8192, 64, 0, 256, 96, False) and not takes(8192, 64, 0, 192, 48, False) and not takes(8192, 256, 0, 256, 64, False)
    assert not takes(8192, 60, 0, 256, 64, False) and not takes(8192, 64, 0, 256, 64, False, gap=4) and not takes(8192, 64, 0, 512, 128, False)

    def longer(f, s):
        s.lda += 8

    def layout(f, s):
        s.b_layout, s.ldb = 1, 256

    def floats(f, s):
        s.out_dtype = s.c_dtype = hk.F32

    def rows(f, s):
        s.init_row_stride, s.init_col_stride = 1, 0

    def tile(f, s):
        f.flags = hk.flag_tile('64x64')

    def strided(f, s):
        f.a2_stride, f.a2_h, f.a2_w, f.a2_oh, f.a2_ow = 2, 128, 256, 64, 128
    for change in (longer, layout, floats, rows, tile):
        assert not takes(8192, 64, 0, 256, 64, False, change=change)
    assert takes(8192, 64, 64, 256, 64, False) and not takes(8192, 64, 64, 256, 64, False, change=strided)


@pytest.mark.gpu
@pytest.mark.parametrize('options,chained', [('hip', True), ('hip{tile=64x64}', False), ('hip{specialise=0,fuse=0}', False)])
def test_residual_blocks_as_a_program(options, chained):
    """Two residual blocks of 1x1 convolutions: the sum is read by the product behind it, by the next residual and by the caller."""
    rng = np.random.default_rng(9)
    W = [E.round_bf16((rng.standard_normal(s) * 0.1).astype(np.float32)) for s in ((1, 1, 64, 256), (1, 1, 256, 64), (1, 1, 64, 256), (1, 1, 256, 128))]
    b = [E.round_bf16(rng.standard_normal(s).astype(np.float32)) for s in (256, 64, 256, 128)]
    X = E.round_bf16(rng.standard_normal((2, 48, 47, 64)).astype(np.float32))
    R = E.round_bf16(rng.standard_normal((2, 48, 47, 256)).astype(np.float32))

    def program(M, O):
        dt = M.DType.BFLOAT16
        x, r = M.Placeholder(dt, X.shape), M.Placeholder(dt, R.shape)
        w, c = [M.Constant(v, dt) for v in W], [M.Constant(v, dt) for v in b]
        y = O.relu(O.convolution(x, w[0]) + c[0] + r)
        t = O.relu(O.convolution(y, w[1]) + c[1])
        z = O.relu(O.convolution(t, w[2]) + c[2] + y)
        return M.Program('blocks', [x, r], [y, z, O.relu(O.convolution(z, w[3]) + c[3])])

    prog = program(P, Pop)
    runner = P.Runner(prog, target=options)
    plan = [v for k, v in prog.passes if k == 'hip-plan'][0]
    assert plan.count('rows multiplied onward') == (2 if chained else 0), plan
    want = E.run(program(E, Eop), [X, R])
    for _ in range(4):  # (the third run records the launches)
        for got, ref in zip(runner.run([X, R]), want):
            np.testing.assert_allclose(got, ref, rtol=2e-2, atol=2e-2)

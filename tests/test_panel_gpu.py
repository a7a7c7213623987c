"""bf16 products over packed right-hand sides in panels (csrc/panel.hip): whole numbers, so that every result is compared value for
value with numpy; rows, columns and K that end inside a tile, a wavefront's blocks, a slab; every configuration that is built."""
import ctypes

import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


def desc(m, n, k, k2=0, mode='plain', gap=0, relu=True, lda_gap=0, stride=0, image=None):
    g = hk.GemmDesc()
    g.in_dtype = g.out_dtype = g.c_dtype = hk.BF16
    g.m, g.n, g.k, g.lda, g.ldb, g.ldc = m, n, k, k + lda_gap, n, n + gap
    g.init_kind, g.init_dtype, g.init_row_stride, g.init_col_stride = int(mode != 'scale'), hk.BF16, 0, 1
    if k2:
        g.k2, g.lda2, g.ldb2, g.init2_kind = k2, k2 + lda_gap, n, 1
        if stride:
            g.a2_stride, g.a2_h, g.a2_w, g.a2_oh, g.a2_ow = (stride,) + image
    ops, operands = {'plain': ([], []),
                     'residual': ([(hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 0, 0.0)], [(hk.BF16, n + gap, 1)]),
                     'scale': ([(hk.EPI_MUL, hk.BF16, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 1, 0.0)], [(hk.BF16, 0, 1)] * 2)}[mode]
    g.tail = hk.make_tail(ops=ops + ([(hk.EPI_RELU, hk.BF16, 0, 0, 0.0)] if relu else []), operands=operands)
    return g


def text_of(g):
    hk.init(0)
    p = hk.lib().pml_hip_gemm_dispatch(ctypes.byref(g))
    assert p, hk.lib().pml_hip_last_error()
    s = hk.describe(p)
    hk.lib().pml_hip_plan_free(p)
    return s


# (m, n, k, what the description says of the panel's tile)
SHAPES = [(21353, 650, 304, '96x768'), (8424, 1805, 312, '192x384'), (7483, 1728, 360, '128x512'), (7059, 1360, 360, '112x512'), (18202, 516, 424, '224x256'),
          (21950, 174, 592, '112x256'), (4424, 1050, 544, '64x512'), (3001, 705, 520, '64x256'), (4095, 1023, 1032, '64x256')]


def run(m, n, k, tile, k2=0, mode='plain', gap=0, lda_gap=0, relu=True, stride=0, image=None, offset=0, packed=True):
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    rng = np.random.default_rng(m + n + k + k2)

    def whole(rows, cols, top=2):
        return rng.integers(-top, top + 1, (rows, cols)).astype(np.float32)
    images = m // (image[2] * image[3]) if stride else 0
    rows2 = images * image[0] * image[1] if stride else m
    A, B = whole(m, k + lda_gap), whole(k, n, 1)
    A2, B2 = whole(rows2, max(k2, 1) + lda_gap), whole(max(k2, 1), n, 1)
    R, b, b2 = whole(m, n + gap, 30), whole(1, n, 9)[0], whole(1, n, 9)[0]
    S, Z = 2.0 ** rng.integers(-2, 3, n).astype(np.float32), whole(1, n, 9)[0]
    A[5, 3], A[m - 1, 0] = np.nan, np.inf
    g = desc(m, n, k, k2, mode, gap, relu, lda_gap, stride, image)
    p = L.pml_hip_gemm_dispatch(ctypes.byref(g))
    assert p, L.pml_hip_last_error()
    assert 'in panels tile=' + tile in hk.describe(p), hk.describe(p)
    dA, dA2, dB, dB2, dR, dS, dZ = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, A2, B, B2, R, S, Z))
    pad = np.full(offset // 2, 77, np.uint16)
    db, db2 = (hk.DeviceBuffer.from_numpy(np.concatenate([pad, T.bf16(x)])) for x in (b, b2))
    dC = hk.DeviceBuffer.from_numpy(np.full(offset // 2 + (m + 1) * (n + gap), 77, np.uint16))
    at = lambda buf: ctypes.c_void_p(int(getattr(buf.ptr, 'value', buf.ptr)) + offset)
    if packed:
        hk.check(L.pml_hip_gemm_pack_b(p, dB.ptr, None))
    if k2:
        hk.check(L.pml_hip_gemm_pack_b2(p, dB2.ptr, None))
    ops = {'plain': none, 'residual': hk.ptr_array([dR.ptr]), 'scale': hk.ptr_array([dS.ptr, dZ.ptr])}[mode]
    for _ in range(2):
        init = at(db) if mode != 'scale' else None
        if k2:
            hk.check(L.pml_hip_gemm_invoke2(p, dA.ptr, None, at(dC), init, dA2.ptr, None, at(db2), ops, none, None))
        else:
            hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, None if packed else dB.ptr, at(dC), init, ops, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(p)
    C = dC.to_numpy(np.uint16, (offset // 2 + (m + 1) * (n + gap),))[offset // 2:].reshape(m + 1, n + gap)
    assert (C[m] == 77).all() and (C[:m, n:] == 77).all()
    a2 = A2[:, :k2]
    if stride:
        a2 = A2.reshape(images, image[0], image[1], -1)[:, ::stride, ::stride, :k2][:, :image[2], :image[3]].reshape(m, k2)
    with np.errstate(invalid='ignore'):
        want = A[:, :k] @ B + (b if mode != 'scale' else 0) + (a2 @ B2 + b2 if k2 else 0)
        want = E.round_bf16(want.astype(np.float32))
        if mode == 'residual':
            want = E.round_bf16(want + R[:, :n])
        if mode == 'scale':
            want = E.round_bf16(E.round_bf16(want * S) + Z)
        if relu:
            want = np.where(want < 0, 0, want)
    np.testing.assert_array_equal(E.bf16_from_bits(C[:m, :n]), want)


@pytest.mark.parametrize('m,n,k,tile', SHAPES)
@pytest.mark.parametrize('mode', ['plain', 'residual', 'scale'])
def test_products(m, n, k, tile, mode):
    if mode != 'plain' and n % 8:
        n = n // 8 * 8
    run(m, n, k, tile if mode == 'plain' else '', mode=mode, gap=8 if n % 8 == 0 else 3, lda_gap=8, relu=mode != 'residual')


@pytest.mark.parametrize('m,n,k,tile', SHAPES)
def test_a_second_product(m, n, k, tile):
    k1 = k // 24 * 8
    run(m, n, k1, '', k2=k - k1, lda_gap=16, mode='plain')
    run(m // 56 * 56, n // 8 * 8, k1, '', k2=k - k1, mode='plain', stride=2, image=(13, 15, 7, 8))


@pytest.mark.parametrize('m,n,k,tile', SHAPES)
def test_right_hand_sides_that_come_with_the_call(m, n, k, tile):
    run(m, n, k, tile, lda_gap=8, packed=False)
    run(m, n // 8 * 8, k, '', mode='residual', packed=False)


@pytest.mark.parametrize('n,gap,offset', [(1000, 0, 0), (1000, 0, 2), (1001, 0, 0), (1001, 7, 6), (993, 0, 16), (999, 1, 4)])
def test_results_anywhere(n, gap, offset):
    run(4100, n, 776, '', gap=gap, offset=offset)


@pytest.mark.parametrize('m,n,k,requantised', [(25089, 512, 1040, False), (9001, 1002, 1040, False), (8424, 1805, 656, True), (16280, 650, 1136, True), (20001, 142, 576, True),
                                               (4093, 3000, 528, True), (11841, 704, 672, True), (19906, 767, 832, True)])
@pytest.mark.parametrize('init,one_scale,offset,packed', [(False, False, 0, True), (True, True, 4, True), (True, False, 16, False)])
def test_int8(m, n, k, requantised, init, one_scale, offset, packed):
    """Sums that wrap past 32 bits among them; value for value."""
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    rng = np.random.default_rng(m + n + k)
    A, B = (rng.integers(-128, 128, s).astype(np.int8) for s in ((m, k), (k, n)))
    b = rng.integers(-2 ** 31, 2 ** 31, n).astype(np.int32) if not requantised else rng.integers(-9000, 9000, n).astype(np.int32)
    S = rng.uniform(0.0001, 0.0006, 1 if one_scale else n).astype(np.float32)
    g = hk.GemmDesc()
    g.in_dtype, g.out_dtype, g.c_dtype = hk.I8, hk.I32, hk.I8 if requantised else hk.I32
    g.m, g.n, g.k, g.lda, g.ldb, g.ldc = m, n, k, k + 16, n, n
    if init:
        g.init_kind, g.init_dtype, g.init_row_stride, g.init_col_stride = 1, hk.I32, 0, 1
    if requantised:
        g.tail = hk.make_tail(ops=[(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -120.0),
                                   (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0), (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)],
                              operands=[(hk.F32, 0, 0 if one_scale else 1)])
    else:
        g.tail = hk.make_tail(ops=[(hk.EPI_RELU, hk.I32, 0, 0, 0.0)])
    p = L.pml_hip_gemm_dispatch(ctypes.byref(g))
    assert p, L.pml_hip_last_error()
    assert 'in panels' in hk.describe(p), hk.describe(p)
    dA = hk.DeviceBuffer.from_numpy(np.concatenate([A, np.full((m, 16), 55, np.int8)], 1))
    dB, dS = hk.DeviceBuffer.from_numpy(B), hk.DeviceBuffer.from_numpy(S)
    db = hk.DeviceBuffer.from_numpy(np.concatenate([np.zeros(offset // 4, np.int32), b]))
    out = np.int8 if requantised else np.int32
    skip = offset // np.dtype(out).itemsize
    dC = hk.DeviceBuffer.from_numpy(np.full(skip + (m + 1) * n, 77, out))
    if packed:
        hk.check(L.pml_hip_gemm_pack_b(p, dB.ptr, None))
    at = lambda buf: ctypes.c_void_p(int(getattr(buf.ptr, 'value', buf.ptr)) + offset)
    for _ in range(2):
        hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, None if packed else dB.ptr, at(dC), at(db) if init else None, hk.ptr_array([dS.ptr]) if requantised else none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(p)
    C = dC.to_numpy(out, (skip + (m + 1) * n,))[skip:].reshape(m + 1, n)
    assert (C[m] == 77).all()
    sums = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.int64) + (b.astype(np.int64) if init else 0)
    sums = sums.astype(np.uint64).astype(np.uint32).view(np.int32)
    if requantised:
        v = np.clip(sums.astype(np.float32) * S, np.float32(-120), np.float32(127))
        want = np.trunc(v + np.copysign(np.float32(0.5), v)).astype(np.int8)
    else:
        want = np.maximum(sums, 0)
    np.testing.assert_array_equal(C[:m], want)


def test_operands_that_a_panel_does_not_read():
    """An operand off 16 bytes, a right-hand side that comes with the call: the other kernels, the same values."""
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    m, n, k = 4100, 1000, 776
    rng = np.random.default_rng(1)
    A, B, R, b = (rng.integers(-t, t + 1, s).astype(np.float32) for t, s in ((2, (m, k)), (1, (k, n)), (30, (m, n)), (9, (n,))))
    p = L.pml_hip_gemm_dispatch(ctypes.byref(desc(m, n, k, mode='residual')))
    assert 'in panels' in hk.describe(p)
    dA, dB, db = (hk.DeviceBuffer.from_numpy(T.bf16(x)) for x in (A, B, b))
    dR = hk.DeviceBuffer.from_numpy(np.concatenate([np.full(1, 77, np.uint16), T.bf16(R).reshape(-1)]))
    want = np.maximum(E.round_bf16(E.round_bf16(A @ B + b) + R), 0)
    hk.check(L.pml_hip_gemm_pack_b(p, dB.ptr, None))
    aligned = hk.DeviceBuffer.from_numpy(T.bf16(R))
    odd = ctypes.c_void_p(int(getattr(dR.ptr, 'value', dR.ptr)) + 2)
    for B_now, res in ((None, aligned.ptr), (dB.ptr, aligned.ptr), (None, odd), (dB.ptr, odd), (None, aligned.ptr)):
        dC = hk.DeviceBuffer.from_numpy(np.full((m, n), 77, np.uint16))
        hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, B_now, dC.ptr, db.ptr, hk.ptr_array([res]), none, None))
        hk.check(L.pml_hip_stream_sync(None))
        np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (m, n))), want)
    # a right-hand side that came with a call is the one that calls without any multiply by from then on, as it always was
    B3 = np.flip(B, 1).copy()
    dB3 = hk.DeviceBuffer.from_numpy(T.bf16(B3))
    for B_now in (dB3.ptr, None):
        hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, B_now, dC.ptr, db.ptr, hk.ptr_array([aligned.ptr]), none, None))
        hk.check(L.pml_hip_stream_sync(None))
        np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (m, n))), np.maximum(E.round_bf16(E.round_bf16(A @ B3 + b) + R), 0))
    L.pml_hip_plan_free(p)


def test_which_products():
    def panels(*a, change=None, **kw):
        g = desc(*a, **kw)
        if change:
            change(g)
        return 'in panels' in text_of(g)
    assert panels(25088, 512, 1024) and panels(25088, 512, 1024, mode='residual') and panels(25088, 512, 1024, mode='scale')
    assert panels(25088, 168, 1024) and not panels(25088, 160, 1024)
    assert panels(4096, 1000, 264) and not panels(100352, 512, 128)  # (those rows stream)
    assert not panels(300, 1000, 264) and not panels(16, 1024, 1024)

    def layout(g):
        g.b_layout, g.ldb = 1, 1024

    def floats(g):
        g.out_dtype = g.c_dtype = hk.F32

    def rows(g):
        g.init_row_stride, g.init_col_stride = 1, 0

    def tile(g):
        g.flags = hk.flag_tile('128x128')
    for change in (layout, floats, rows, tile):
        assert not panels(25088, 512, 1024, change=change), change


# (the last ones: a right-hand side that fits the array of the entry without a plan to the last bytes, as fragments too, and not as fragments)
@pytest.mark.parametrize('m,n,k,tile', SHAPES + [(2000, 3000, 5568, ''), (2000, 3489, 4808, '')])
def test_the_entry_without_a_plan_gives_the_same_bits(m, n, k, tile):
    """Sums of floats, which another order would round otherwise."""
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    rng = np.random.default_rng(m + n + k)
    g = desc(m, n, k, lda_gap=8)
    p = L.pml_hip_gemm_dispatch(ctypes.byref(g))
    assert 'in panels tile=' + tile in hk.describe(p), hk.describe(p)
    dA, dB, db = (hk.DeviceBuffer.from_numpy(T.bf16(rng.standard_normal(s).astype(np.float32))) for s in ((m, k + 8), (k, n), (n,)))
    dC, dD = (hk.DeviceBuffer.from_numpy(np.full((m, n), 77, np.uint16)) for _ in range(2))
    hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, dB.ptr, dC.ptr, db.ptr, none, none, None))
    hk.check(L.pml_hip_gemm_run_static(ctypes.byref(g), dA.ptr, dB.ptr, dD.ptr, db.ptr, none, none, None))
    hk.check(L.pml_hip_stream_sync(None))
    L.pml_hip_plan_free(p)
    np.testing.assert_array_equal(dC.to_numpy(np.uint16, (m, n)), dD.to_numpy(np.uint16, (m, n)))


def test_texts_name_what_multiplies_a_right_hand_side_that_comes_with_the_call():
    def requantised(m, n, k):
        g = hk.GemmDesc()
        g.in_dtype, g.out_dtype, g.c_dtype = hk.I8, hk.I32, hk.I8
        g.m, g.n, g.k, g.lda, g.ldb, g.ldc = m, n, k, k, n, n
        g.tail = hk.make_tail(ops=[(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -120.0),
                                   (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0), (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)],
                              operands=[(hk.F32, 0, 1)])
        return text_of(g)
    for m, n, k, in_call in ((4096, 4096, 4096, True), (6000, 3200, 3072, True), (4096, 4096, 2048, False), (4096, 4094, 2048, True)):
        text = requantised(m, n, k)
        assert 'with B packed ' + ('ahead or in the call in panels' if in_call else 'in panels') in text and ('with B as it lies' in text) != in_call, text
    for m, n, k, tile in SHAPES:
        text = text_of(desc(m, n, k))
        assert 'with B packed ' + ('in panels' if 'as it lies' in text else 'ahead or in the call in panels') in text and 'packed through' not in text, text


def test_a_packing_that_is_recorded():
    """Into a graph, where nothing may be allocated: by a plan that has no room for fragments yet, and by one that has."""
    hk.init(0)
    L, none = hk.lib(), hk.ptr_array([])
    m = n = k = 4096
    rng = np.random.default_rng(3)
    A, B = rng.integers(-2, 3, (m, k)).astype(np.float32), rng.integers(-1, 2, (k, n)).astype(np.float32)
    g = desc(m, n, k, mode='scale')
    g.tail = hk.make_tail()
    want = E.round_bf16(A @ B)
    dA, dB = hk.DeviceBuffer.from_numpy(T.bf16(A)), hk.DeviceBuffer.from_numpy(T.bf16(B))
    for ahead in (False, True):
        p = L.pml_hip_gemm_dispatch(ctypes.byref(g))
        assert 'with B as it lies through registers' in hk.describe(p) and 'with B packed in panels' in hk.describe(p), hk.describe(p)
        if ahead:
            hk.check(L.pml_hip_gemm_pack_b(p, dA.ptr, None))
            hk.check(L.pml_hip_stream_sync(None))
        stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
        hk.check(L.pml_hip_stream_create(ctypes.byref(stream)))
        hk.check(L.pml_hip_capture_begin(stream))
        rc = L.pml_hip_gemm_pack_b(p, dB.ptr, stream)
        hk.check(L.pml_hip_capture_end(stream, ctypes.byref(graph)))
        hk.check(rc)
        for _ in range(3):
            dC = hk.DeviceBuffer.from_numpy(np.full((m, n), 77, np.uint16))
            hk.check(L.pml_hip_graph_launch(graph, stream))
            hk.check(L.pml_hip_gemm_invoke(p, dA.ptr, None, dC.ptr, None, none, none, stream))
            hk.check(L.pml_hip_stream_sync(stream))
            np.testing.assert_array_equal(E.bf16_from_bits(dC.to_numpy(np.uint16, (m, n))), want)
        L.pml_hip_graph_destroy(graph)
        L.pml_hip_stream_destroy(stream)
        L.pml_hip_plan_free(p)


# every configuration with a second product (K: of both), and for either result of int8 (the 192x384 one is no int32 product's)
SECONDS = [(19945, 193, 272, '112x256'), (2172, 3910, 280, '112x512'), (14793, 614, 296, '128x512'), (13657, 1078, 288, '192x384'),
           (18752, 611, 320, '224x256'), (1281, 202, 1120, '64x256'), (10897, 309, 272, '64x512'), (11923, 1234, 288, '96x768')]
INT8 = [(18633, 130, 1024, False, '112x256'), (23195, 257, 1024, False, '112x512'), (15284, 518, 1024, False, '128x512'), (16714, 600, 1024, False, '224x256'),
        (4030, 919, 1024, False, '64x256'), (11008, 269, 1024, False, '64x512'), (19821, 520, 1024, False, '96x768'), (17666, 141, 528, True, '112x256'),
        (19422, 258, 528, True, '112x512'), (15482, 542, 528, True, '128x512'), (8216, 1778, 528, True, '192x384'), (16714, 600, 528, True, '224x256'),
        (8653, 140, 528, True, '64x256'), (8702, 275, 528, True, '64x512'), (19642, 541, 528, True, '96x768')]


@pytest.mark.parametrize('m,n,k,tile', SECONDS)
def test_every_configuration_with_a_second_product(m, n, k, tile):
    k1 = k // 24 * 8
    run(m, n, k1, tile + ' (', k2=k - k1, lda_gap=16, gap=3)


@pytest.mark.parametrize('m,n,k,requantised,tile', INT8)
def test_every_configuration_int8(m, n, k, requantised, tile):
    g = hk.GemmDesc()
    g.in_dtype, g.out_dtype, g.c_dtype = hk.I8, hk.I32, hk.I8 if requantised else hk.I32
    g.m, g.n, g.k, g.lda, g.ldb, g.ldc = m, n, k, k + 16, n, n
    if requantised:
        g.tail = hk.make_tail(ops=[(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -120.0),
                                   (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0), (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)],
                              operands=[(hk.F32, 0, 1)])
    assert 'in panels tile=%s (' % tile in text_of(g), text_of(g)
    test_int8(m, n, k, requantised, True, False, 4, True)

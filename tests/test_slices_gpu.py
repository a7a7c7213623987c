"""Programs that run in parts of the leading dimension, and runs whose copies and launches overlap (host/src/hip_plan_slice.cc,
hip_runtime.cc): whole numbers, so that every run is compared value for value with numpy."""
import re

import numpy as np
import pytest

from plaidml_amd import edsl as P
from plaidml_amd import op as Pop

DT = {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16}


def whole(rng, *shape, top=2):
    return rng.integers(-top, top + 1, shape).astype(np.float32)


def dense(dt, m, k=640):
    """Operands in parts and as a whole, a product on top of the one in parts."""
    X, R, W, V, b = (P.Placeholder(DT[dt], s) for s in ([m, k], [m, 256], [k, 256], [256, 64], [256]))
    y = Pop.relu(Pop.dot(X, W) + b + R)
    draw = lambda rng: [whole(rng, m, k), whole(rng, m, 256), whole(rng, k, 256, top=1), whole(rng, 256, 64, top=1) * (rng.random((256, 64)) < 0.05), whole(rng, 256)]

    def want(x, r, w, v, c):
        y = np.maximum(x @ w + c + r, 0)
        return [y, y @ v]
    return P.Program('dense', [X, R, W, V, b], [y, Pop.dot(y, V)]), draw, want


def images(dt, n, hw=64):
    """A convolution and a maximum over windows in parts, their sum over images not."""
    X, F = P.Placeholder(DT[dt], [n, hw, hw, 64]), P.Placeholder(DT[dt], [1, 1, 64, 512])
    y = Pop.relu(Pop.convolution(X, F, strides=[1, 1]))
    top = Pop.pool(y, 'max', [2, 2], [2, 2], autopad='valid')
    draw = lambda rng: [whole(rng, n, hw, hw, 64), whole(rng, 1, 1, 64, 512, top=1)]

    def want(x, f):
        return [np.maximum(x.reshape(-1, 64) @ f.reshape(64, 512), 0).reshape(n, hw // 2, 2, hw // 2, 2, 512).max((0, 2, 4))]
    return P.Program('images', [X, F], [Pop.max(top, axes=[0])]), draw, want


def rows(dt, m, c=520):
    X, g = P.Placeholder(DT[dt], [m, c]), P.Placeholder(DT[dt], [c])
    d = X - Pop.max(X, axes=[-1], keepdims=True)
    draw = lambda rng: [whole(rng, m, c, top=60), whole(rng, c)]
    return P.Program('rows', [X, g], [d * g]), draw, lambda x, h: [(x - x.max(-1, keepdims=True)) * h]


def batches(dt, n, r=96):
    A, B = P.Placeholder(DT[dt], [n, r, 64]), P.Placeholder(DT[dt], [n, 64, 80])
    x, i, j, k = P.TensorIndexes(4)
    C = P.Contraction().outShape(n, r, 80).outAccess(x, i, j).sum(A[x, i, k] * B[x, k, j]).build()
    draw = lambda rng: [whole(rng, n, r, 64), whole(rng, n, 64, 80, top=1)]
    return P.Program('batches', [A, B], [C]), draw, lambda a, b: [np.matmul(a, b)]


CASES = {'dense': (dense, 3571), 'dense even': (dense, 4096), 'images': (images, 21), 'rows': (rows, 5003), 'batches': (batches, 401)}


def runs_from(program, target=''):
    program.compile(target)
    m = re.search(r'beside launches ahead of steps? ([0-9, ]+)', dict(program.passes)['hip-plan'])
    return [int(i) for i in m.group(1).split(',')] if m else []


def test_which_launches_copies_go_beside():
    """Long results are followed by a run of launches of its own, long operands where there is enough ahead of them to hide it."""
    i, j, k = P.TensorIndexes(3)

    def result(m):  # of m KB
        A, W, V = (P.Placeholder(DT['f32'], s) for s in ([m, 64], [64, 256], [256, 8]))
        y = Pop.dot(A, W)
        return P.Program('result', [A, W, V], [y, Pop.dot(y, V)])

    def operand(m, launches):  # of m KB behind so many products
        A, B = P.Placeholder(DT['f32'], [128, 128]), P.Placeholder(DT['f32'], [m, 256])
        x = A
        for _ in range(launches):
            x = Pop.relu(Pop.dot(x, A) * (1 / 64))
        return P.Program('operand', [A, B], [P.Contraction().outShape(256, 128).outAccess(i, j).sum(B[k, i] * Pop.dot(P.Constant(whole(np.random.default_rng(1), m, 128), DT['f32']), x)[k, j]).build()])
    assert runs_from(result(4095)) == [] and runs_from(result(4096)) == [1] and runs_from(result(4096), 'hip{overlap=0}') == []
    # (a launch is taken to take 6 us, 60 have to lie ahead)
    assert runs_from(operand(8192, 2)) == [] and runs_from(operand(8192, 12)) == [13] and runs_from(operand(4095, 12)) == []
    A, B, V = (P.Placeholder(DT['f32'], s) for s in ([23, 17, 128], [23, 370, 128], [23, 370, 128]))
    x, i, j, k = P.TensorIndexes(4)
    S = Pop.softmax(P.Contraction().outShape(23, 17, 370).outAccess(x, i, j).sum(A[x, i, k] * B[x, j, k]).build(), -1)
    assert runs_from(P.Program('batched', [A, B, V], [P.Contraction().outShape(23, 17, 128).outAccess(x, i, k).sum(S[x, i, j] * V[x, j, k]).build()])) == []


def build(name, dt, scale=1):
    fn, size = CASES[name]
    return fn(dt, size * scale)


def parts(program):
    program.compile('')
    m = re.search(r'steps 0 to (\d+) in (\d+) parts', dict(program.passes)['hip-plan'])
    return (int(m.group(1)) + 1, int(m.group(2))) if m else (0, 1)


def test_what_runs_in_parts():
    for name in CASES:
        steps, n = parts(build(name, 'f32')[0])
        assert steps >= 1 and 2 <= n <= 4, name
        assert n == 2, name
    assert parts(dense('f32', 64)[0]) == (0, 1)  # (nothing to carry meanwhile)
    assert parts(batches('f32', 150)[0]) == (0, 1) and parts(batches('f32', 220)[0])[1] == 2  # (parts of 4 MB and more)
    X, W = P.Placeholder(DT['f32'], [4096, 1024]), P.Placeholder(DT['f32'], [4096, 64])
    i, j, k = P.TensorIndexes(3)
    # rows of the result are columns of what comes in
    assert parts(P.Program('across', [X, W], [P.Contraction().outShape(1024, 64).outAccess(i, j).sum(X[k, i] * W[k, j]).build()])) == (0, 1)
    # the same value in parts and as a whole
    S = P.Placeholder(DT['f32'], [2048, 2048])
    assert parts(P.Program('square', [S], [Pop.dot(S, S)])) == (0, 1)
    # sums over the leading dimension
    assert parts(P.Program('sum', [X], [Pop.sum(X, axes=[0])])) == (0, 1)


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('pinned_results', [True, False])
@pytest.mark.parametrize('name', sorted(CASES))
def test_every_run(monkeypatch, dt, pinned_results, name):
    """Launched one by one, recorded and replayed; whole runs with other values each time; a profile and no page-locked memory between."""
    print(name, dt, flush=True)
    if not pinned_results:
        monkeypatch.setattr(P, '_result_array', lambda d, sizes, nbytes: np.empty(sizes, d))
    program, draw, want = build(name, dt, 1 if dt == 'f32' else 2)
    if name == 'dense':
        assert parts(program)[1] > 1
    steps, n = parts(program)
    launches = int(re.search(r'(\d+) launches', dict(program.passes)['hip-plan']).group(1)) + steps * (n - 1)
    runner = P.Runner(program, target='hip')
    rounded = (lambda a: a) if dt == 'f32' else P.round_bf16
    for run in range(7):
        arrays = draw(np.random.default_rng(run))
        with monkeypatch.context() as patch:
            if run == 4:
                patch.setenv('PLAIDML_PROFILE', '1')
            if run == 5:
                patch.setenv('PLAIDML_PINNED', '0')
            got = runner.run(arrays)
        s = P.last_run_stats()
        assert s['kernel_ms'] > 0 and s['h2d_ms'] + s['kernel_ms'] + s['d2h_ms'] == pytest.approx(runner.ms, rel=1e-6, abs=1e-9)
        assert s['launches'] == launches
        exact = want(*arrays)
        if name.startswith('dense') and dt == 'bf16':  # (the second product takes the rounded first one)
            exact = [exact[0], rounded(exact[0]) @ arrays[3]]
        for k, (g, w) in enumerate(zip(got, exact)):
            np.testing.assert_array_equal(g, rounded(w.astype(np.float32)), err_msg='%s run %d result %d' % (name, run, k))


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('pinned_results', [True, False])
def test_more_than_the_staging_holds(monkeypatch, dt, pinned_results):
    """Operands past the staging's slots, of which every part takes several, and results that come back through them."""
    if not pinned_results:
        monkeypatch.setattr(P, '_result_array', lambda d, sizes, nbytes: np.empty(sizes, d))
    m = {'f32': 18001, 'bf16': 36001}[dt]  # 46 MB
    program, draw, want = dense(dt, m)
    assert parts(program)[1] > 1
    runner = P.Runner(program, target='hip')
    for run in range(5):
        arrays = draw(np.random.default_rng(run))
        got = runner.run(arrays)
        exact = want(*arrays)
        if dt == 'bf16':
            exact = [P.round_bf16(exact[0]), P.round_bf16(P.round_bf16(exact[0]) @ arrays[3])]
        for g, w in zip(got, exact):
            np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['f32', 'bf16'])
def test_results_over_operands(dt):
    """A result in the memory of an operand that a later launch, or a later part of the same one, is the first to need."""
    m = 2048 if dt == 'f32' else 4096
    bits = (lambda a: a) if dt == 'f32' else P.to_bf16_bits
    value = (lambda a: a) if dt == 'f32' else P.from_bf16_bits
    rounded = (lambda a: a) if dt == 'f32' else P.round_bf16
    i, j, k = P.TensorIndexes(3)
    A, W, B, V = (P.Placeholder(DT[dt], s) for s in ([m, 1024], [1024, 1024], [m, 1024], [m, 64]))
    second = P.Contraction().outShape(1024, 64).outAccess(i, j).sum(B[k, i] * V[k, j]).build()
    two = P.Runner(P.Program('two', [A, W, B, V], [Pop.dot(A, W), second]), target='hip')
    X, U = P.Placeholder(DT[dt], [m, 512]), P.Placeholder(DT[dt], [512, 1024])
    program = P.Program('longer', [X, U], [Pop.relu(Pop.dot(X, U))])
    assert parts(program)[1] == 2  # (rows of the result reach further than those of the operand)
    longer = P.Runner(program, target='hip')
    for run in range(6):
        rng = np.random.default_rng(run)
        a, w, b, v = whole(rng, m, 1024), whole(rng, 1024, 1024, top=1), whole(rng, m, 1024), whole(rng, m, 64, top=1)
        staged = two.stage([a, w, b, v])
        two.exe.run(staged, [staged[2], two.outputs[1]])
        np.testing.assert_array_equal(value(staged[2].as_ndarray()), rounded(a @ w), err_msg='run %d' % run)
        np.testing.assert_array_equal(value(two.outputs[1].as_ndarray()), rounded(b.T @ v), err_msg='run %d' % run)
        x, u = whole(rng, m, 512), whole(rng, 512, 1024, top=1)
        memory = P._result_array(np.dtype(np.float32 if dt == 'f32' else np.uint16), (m, 1024), m * 1024 * (4 if dt == 'f32' else 2))
        operand, result = P.Buffer(longer.in_shapes[0], data=memory[:m // 2].reshape(m, 512)), P.Buffer(longer.out_shapes[0], data=memory)
        operand.copy_from_ndarray(bits(x))
        longer.exe.run([operand, longer.stage([x, u])[1]], [result])
        np.testing.assert_array_equal(value(memory), rounded(np.maximum(x @ u, 0)), err_msg='run %d' % run)


@pytest.mark.gpu
def test_launches_ahead_of_every_operand():
    """Launches that need no operand run while operands travel, and their time counts."""
    one = lambda *shape: np.full(shape, 0.5, np.float32)
    bf = P.DType.BFLOAT16
    c, d = P.Constant(one(4096, 4096), bf), P.Constant(one(4096, 4096), bf)
    X, V = P.Placeholder(bf, [4096, 4096]), P.Placeholder(bf, [4096, 64])
    program = P.Program('ahead', [X, V], [Pop.dot(c, d), Pop.dot(X, V)])
    runner = P.Runner(program, target='hip')
    plan = dict(program.passes)['hip-plan']
    assert '2 launches' in plan and plan.index('k=4096 B=[k][n]') < plan.index('n=64'), plan
    for run in range(4):
        rng = np.random.default_rng(run)
        x, v = whole(rng, 4096, 4096), whole(rng, 4096, 64, top=1)
        got = runner.run([x, v])
        s = P.last_run_stats()
        # 137 GFLOP at the 2.5 PFLOP/s the device has at most
        assert s['launches'] == 2 and s['kernel_ms'] > 0.055, s
        assert (got[0] == 1024).all()
        np.testing.assert_array_equal(got[1], P.round_bf16(x @ v))


@pytest.mark.gpu
@pytest.mark.parametrize('n, hw, ci, co', [(10, 49, 117, 26), (3, 106, 52, 19)])
def test_copies_up_do_not_wait_for_copies_down(n, hw, ci, co):
    """Both gradients of a 5x5 convolution, X needed by the second launch only and as long as the first one's result: the one goes up
    beside the other, whichever copy engines the two are given (the process's other streams decide that).

    One stream: all up, both launches, all down, of which X's way up or the result's is a quarter and more; half of that is asked for
    (measured 0.70 and 0.74 of the one stream's time; 1.02 and 1.03 where X waited behind a result that waited for its launch)."""
    import torch
    torch.zeros(1, device='cuda')
    X, F, G = (P.Placeholder(DT['f32'], s) for s in ([n, hw, hw, ci], [5, 5, ci, co], [n, hw, hw, co]))
    program = P.Program('gradients', [X, F, G], [Pop.convolution(G, F, strides=[1, 1], deriv_mode=Pop.DERIV_DATA, result_shape=[hw, hw]),
                                                 Pop.convolution(X, G, strides=[1, 1], deriv_mode=Pop.DERIV_FILTER, result_shape=[5, 5])])
    runners = P.Runner(program, target='hip'), P.Runner(program, target='hip{overlap=0}')
    rng = np.random.default_rng(3)
    arrays = [whole(rng, n, hw, hw, ci, top=1), whole(rng, 5, 5, ci, co, top=1), whole(rng, n, hw, hw, co, top=1)]
    times, got = ([], []), [None, None]
    for block in range(9):
        for which in (0, 1) if block % 2 else (1, 0):
            for _ in range(6):
                got[which] = runners[which].run(arrays)
                if block:
                    times[which].append(runners[which].ms)
    for g, w in zip(*got):  # (whole numbers below 2^24, whatever the order of sums)
        np.testing.assert_array_equal(g, w)
    beside, behind = (np.median(t) for t in times)
    print('%d x %d x %d x %d -> %d: beside %.3f ms, behind %.3f ms' % (n, hw, hw, ci, co, beside, behind), flush=True)
    assert beside < 0.88 * behind


@pytest.mark.gpu
def test_launches_do_not_wait_for_copies_down():
    """A long result goes down beside the launches behind it, also where a run's streams share a queue of the device: streams are
    made in fours and one of each four is given up, so that the run's three come to where it was.

    Of the one stream's time the small launches take a fifth, which the result hides (measured 0.86 to 0.89 of it; 1.24 with the
    launches behind the copy, which is what waiting between streams costs besides)."""
    import ctypes
    import torch
    from plaidml_amd import hipkernels as hk
    torch.zeros(1, device='cuda')
    hk.init(0)
    A, W, V = (P.Placeholder(DT['f32'], s) for s in ([1024, 64], [64, 1024], [1024, 8]))
    y = Pop.dot(A, W)
    program = P.Program('result', [A, W, V], [y, Pop.dot(Pop.sum(y, axes=[0], keepdims=True), V)])
    rng = np.random.default_rng(4)
    arrays = [whole(rng, 1024, 64), whole(rng, 64, 1024), whole(rng, 1024, 8)]
    want = [arrays[0] @ arrays[1], (arrays[0] @ arrays[1]).sum(0, keepdims=True) @ arrays[2]]

    def median(runner):
        times = []
        for run in range(40):
            got = runner.run(arrays)
            if run >= 8:
                times.append(runner.ms)
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, w)
        return np.median(times)
    behind = median(P.Runner(program, target='hip{overlap=0}'))
    for place in range(4):
        streams = [ctypes.c_void_p() for _ in range(16)]
        for s in streams:
            hk.check(hk.lib().pml_hip_stream_create(ctypes.byref(s)))
        for s in streams[place::4]:
            hk.check(hk.lib().pml_hip_stream_destroy(s))
        beside = median(P.Runner(program, target='hip'))
        for s in (s for k, s in enumerate(streams) if k % 4 != place):
            hk.check(hk.lib().pml_hip_stream_destroy(s))
        print('place %d: beside %.3f ms, behind %.3f ms' % (place, beside, behind), flush=True)
        assert beside < behind


@pytest.mark.gpu
@pytest.mark.parametrize('name', ['dense', 'images', 'batches'])
def test_the_option_that_keeps_steps_whole(name):
    program, draw, want = build(name, 'f32')
    assert parts(program)[1] == 2
    program.compile('hip{overlap=0}')
    assert 'parts' not in dict(program.passes)['hip-plan']
    runner = P.Runner(program, target='hip{overlap=0}')
    launches = int(re.search(r'(\d+) launches', dict(program.passes)['hip-plan']).group(1))
    for run in range(4):
        arrays = draw(np.random.default_rng(run))
        for g, w in zip(runner.run(arrays), want(*arrays)):
            np.testing.assert_array_equal(g, w.astype(np.float32))
        assert P.last_run_stats()['launches'] == launches


# Every kind of step that is cut, with a shorter last part and rows or images that begin anywhere in their part: (program, draws,
# what its plan says).  Whole numbers or one and the same kernel: a run on whole steps gives the same bits.
def softmax(dt, m, c=1001):
    X = P.Placeholder(DT[dt], [m, c])
    return P.Program('softmax', [X], [Pop.softmax(X, -1), Pop.argmax(X, 1)]), lambda rng: [whole(rng, m, c, top=9)], ['softmax', 'argmax']


def topk(dt, m, c=1001):
    X = P.Placeholder(DT[dt], [m, c])
    return P.Program('topk', [X], [Pop.softmax(X, -1)] + list(Pop.topk(X, 5))), lambda rng: [whole(rng, m, c, top=9)], ['softmax', 'top 5']


def rows_with_scalars(dt, m, c=1001):
    X, s, g = (P.Placeholder(DT[dt], sizes) for sizes in ([m, c], [m, 1], [c]))
    top = Pop.max(X, 1, True)
    return P.Program('scalars', [X, s, g], [(X - top) * s + g, top * s]), lambda rng: [whole(rng, m, c), whole(rng, m, 1, top=9), whole(rng, c)], ['row program']


def odd_batches(dt, n, r=97):
    A, B = P.Placeholder(DT[dt], [n, r, 63]), P.Placeholder(DT[dt], [n, 63, 81])
    x, i, j, k = P.TensorIndexes(4)
    C = P.Contraction().outShape(n, r, 81).outAccess(x, i, j).sum(A[x, i, k] * B[x, k, j]).build()
    return P.Program('batches', [A, B], [C]), lambda rng: [whole(rng, n, r, 63), whole(rng, n, 63, 81, top=1)], ['97']


def odd_rows(dt, m, k=1003):
    """(K off whole vectors: a product over free strides)"""
    X, W, b = P.Placeholder(DT[dt], [m, k]), P.Placeholder(DT[dt], [k, 1001]), P.Placeholder(DT[dt], [1001])
    return P.Program('rows', [X, W, b], [Pop.relu(Pop.dot(X, W) + b)]), lambda rng: [whole(rng, m, k), whole(rng, k, 1001, top=1), whole(rng, 1001)], ['product']


def few_channels(dt, n, stride=1, h=63, w=61, co=7):
    X, F, b = P.Placeholder(DT[dt], [n, h, w, 3]), P.Placeholder(DT[dt], [5, 5, 3, co]), P.Placeholder(DT[dt], [co])
    y = Pop.relu(Pop.convolution(X, F, strides=[stride] * 2) + b)
    return P.Program('channels', [X, F, b], [y]), lambda rng: [whole(rng, n, h, w, 3), whole(rng, 5, 5, 3, co, top=1), whole(rng, co)], ['conv2d']


def stem(dt, n):
    return few_channels(dt, n, stride=2, co=64)


def pooled_stem(dt, n, hw=128):
    """(in bf16 the convolution pools inside its launch)"""
    X = P.Placeholder(DT[dt], [n, hw, hw, 3])
    rng = np.random.default_rng(6)
    F, b = P.Constant(whole(rng, 7, 7, 3, 64, top=1), DT[dt]), P.Constant(whole(rng, 64), DT[dt])
    y = Pop.relu(Pop.convolution(X, F, strides=[2, 2], autopad=Pop.SAME_UPPER) + b)
    text = '+ max-pool 3x3 stride 2' if dt == 'bf16' else 'pool2d max'
    return P.Program('stem', [X], [Pop.pool(y, 'max', [3, 3], [2, 2], autopad=Pop.SAME_UPPER)]), lambda rng: [whole(rng, n, hw, hw, 3)], [text]


def depthwise(dt, n, hw=33, c=72):
    X, F = P.Placeholder(DT[dt], [n, hw, hw, c]), P.Placeholder(DT[dt], [3, 3, c, 1])
    y = Pop.relu(Pop.convolution(X, F, depthwise=True))
    return P.Program('depthwise', [X, F], [y]), lambda rng: [whole(rng, n, hw, hw, c), whole(rng, 3, 3, c, 1)], ['dwconv2d']


def separable(dt, n, hw=19, c=104):
    """Depthwise, pointwise with scale and shift, maximum and its place in the window."""
    X = P.Placeholder(DT[dt], [n, hw, hw, c])
    rng = np.random.default_rng(4)
    F, W, s, z = (P.Constant(v, DT[dt]) for v in (whole(rng, 3, 3, c, 1), whole(rng, 1, 1, c, c, top=1), 2.0 ** whole(rng, c, top=1), whole(rng, c)))
    R = Pop.relu(Pop.convolution(Pop.convolution(X, F, depthwise=True), W) * s + z)
    M = Pop.pool(R, 'max', [3, 3], [2, 2], autopad=Pop.SAME_UPPER)
    b, x0, x1, ch, k0, k1 = P.TensorIndexes(6)
    IX = P.index([3, 3], 0) * 3 + P.index([3, 3], 1)
    AM = P.Contraction().outShape(M.shape).outAccess(b, x0, x1, ch).max(P.cond(R[b, 2 * x0 + k0 - 1, 2 * x1 + k1 - 1, ch], M[b, x0, x1, ch], IX[k0, k1])).build()
    return P.Program('separable', [X], [R, M, AM]), lambda rng: [whole(rng, n, hw, hw, c)], ['dwconv2d', 'pool2d']


def blocks(dt, n, hw=47, stride=1):
    """A residual block behind a projection of its own rows, and the product that the chip multiplies its rows onward to (bf16)."""
    side = (hw - 1) // stride + 1
    X, T = P.Placeholder(DT[dt], [n, hw, hw, 64]), P.Placeholder(DT[dt], [n, side, side, 64])
    rng = np.random.default_rng(5)
    w, v, u = (P.Constant(whole(rng, 1, 1, *s, top=1) * (rng.random(s) < 0.2), DT[dt]) for s in ((64, 256), (64, 256), (256, 64)))
    c, d = (P.Constant(whole(rng, k), DT[dt]) for k in (256, 256))
    y = Pop.relu(Pop.convolution(T, w) + c + (Pop.convolution(X, v, strides=[stride] * 2) + d))
    draw = lambda rng: [whole(rng, n, hw, hw, 64), whole(rng, n, side, side, 64, top=1)]
    return P.Program('blocks', [X, T], [y, Pop.relu(Pop.convolution(y, u))]), draw, ['second product'] if dt == 'bf16' else []


def strided_blocks(dt, n):
    return blocks(dt, n, hw=113, stride=2)


# (odd numbers of rows or images, of which the first part has an odd number too)
KINDS = {f.__name__: (f, sizes) for f, *sizes in ((softmax, 4001, 8001), (topk, 4001, 8001), (rows_with_scalars, 4001, 8001), (odd_batches, 401, 801), (odd_rows, 4001, 8001),
                                                  (few_channels, 201, 405), (stem, 201, 405), (pooled_stem, 81, 161), (depthwise, 61, 121), (separable, 61, 121), (blocks, 29, 29), (strided_blocks, 21, 21))}


def kind(name, dt):
    fn, (f32, bf16) = KINDS[name]
    return fn(dt, f32 if dt == 'f32' else bf16)


@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('name', sorted(KINDS))
def test_which_kinds_run_in_parts(dt, name):
    """All of the program, in two parts, the second one shorter."""
    program, _, texts = kind(name, dt)
    steps, n = parts(program)
    plan = dict(program.passes)['hip-plan']
    assert n == 2 and '%d launches' % steps in plan and all(t in plan for t in texts), plan
    assert all(size % 4 == 1 for size in KINDS[name][1])


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('name', sorted(KINDS))
def test_every_kind_of_step(dt, name):
    print(name, dt, flush=True)
    program, draw, _ = kind(name, dt)
    assert parts(program)[1] == 2
    cut, whole_steps = P.Runner(program, target='hip'), P.Runner(program, target='hip{overlap=0}')
    for run in range(4):
        arrays = draw(np.random.default_rng(run))
        for k, (g, w) in enumerate(zip(cut.run(arrays), whole_steps.run(arrays))):
            assert np.any(w) and g.dtype == w.dtype
            np.testing.assert_array_equal(g, w, err_msg='%s run %d result %d' % (name, run, k))

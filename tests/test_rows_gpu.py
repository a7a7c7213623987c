"""Operations along the last axis in one launch (csrc/rows.hip): normalisations as row programs, argmax, the first k of a sort, against
numpy; row lengths around a wavefront's and a workgroup's width, ties and NaNs."""
import numpy as np
import pytest

from plaidml_amd import edsl as P
from plaidml_amd import op as Pop

pytestmark = pytest.mark.gpu
DT = {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16, 'i32': P.DType.INT32, 'u8': P.DType.UINT8}
SHAPES = [(1, 2), (3, 63), (5, 256), (4, 257), (2, 512), (7, 513), (1, 1000), (9, 2049), (2, 7999), (2, 3, 5, 100)]


def run(make, arrays, dtype, text):
    inputs = [P.Placeholder(DT[dtype], a.shape) for a in arrays]
    program = P.Program('rows', inputs, make(*inputs))
    runner = P.Runner(program, target='hip')
    for _ in range(4):  # one by one, then (for programs of several launches) as a recorded graph
        got = runner.run(arrays)
    plan = [v for k, v in program.passes if k == 'hip-plan'][0]
    assert text in plan and '1 launches' in plan, plan
    return got


def values(rng, shape, dtype):
    if dtype == 'i32':
        return rng.integers(-5, 6, shape, dtype=np.int32) * 400000000
    if dtype == 'u8':
        return rng.integers(0, 256, shape, dtype=np.uint8)
    a = rng.standard_normal(shape).astype(np.float32)
    return P.round_bf16(a) if dtype == 'bf16' else a


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('shape', SHAPES)
def test_normalised_rows(dtype, shape):
    rng = np.random.default_rng(shape[-1])
    x, g, s = values(rng, shape, dtype) * 2 + 1, values(rng, shape[-1:], dtype), values(rng, shape[-1:], dtype)
    if dtype == 'bf16':
        x = P.round_bf16(x)
    got, = run(lambda X, G, S: [Pop.mvn(X, axes=[len(shape) - 1]) * G + S], [x, g, s], dtype, 'row program')
    x64 = x.astype(np.float64)
    c = x64 - x64.mean(-1, keepdims=True)
    want = c / np.maximum(np.sqrt((c * c).mean(-1, keepdims=True)), 1e-9) * g + s
    assert np.linalg.norm(got - want) < (2e-2 if dtype == 'bf16' else 2e-6) * np.linalg.norm(want)


def test_row_program_with_several_results():
    rng = np.random.default_rng(3)
    x, r = values(rng, (6, 130), 'f32'), values(rng, (6, 1), 'f32')

    def make(X, R):
        m = Pop.max(X, 1, True)
        e = P.exp(X - m) * R
        s = Pop.sum(e, 1, True)
        return [s * 2.0, (e / s) + X, -m]
    s, q, m = run(make, [x, r], 'f32', 'row program')
    we = np.exp(x - x.max(1, keepdims=True)) * r
    np.testing.assert_allclose(s, 2 * we.sum(1, keepdims=True), rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(q, we / we.sum(1, keepdims=True) + x, rtol=1e-4, atol=1e-4)
    np.testing.assert_array_equal(m, -x.max(1, keepdims=True))


@pytest.mark.parametrize('rows,cols', [(1024, 1500), (1024, 2016), (1025, 2020), (1030, 2048)])
def test_row_program_with_many_live_vectors(rows, cols):
    """Five values per column are live at once: four rows of up to 2016 columns share a workgroup's LDS, longer ones have it alone."""
    x = values(np.random.default_rng(cols), (rows, cols), 'f32')

    def make(X):
        t = X - Pop.max(X, 1, True)
        a, b = P.exp(t), P.tanh(t)
        c, d = a * b, b * b
        sums = [Pop.sum(v, 1, True) for v in (a, b, c, d)]
        return [a / sums[0] + b / sums[1] + c / sums[2] + d / sums[3] + t]
    got, = run(make, [x], 'f32', 'row program')
    t = x.astype(np.float64) - x.max(1, keepdims=True)
    a, b = np.exp(t), np.tanh(t)
    want = sum(v / v.sum(1, keepdims=True) for v in (a, b, a * b, b * b)) + t
    assert np.linalg.norm(got - want) < 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('shape', SHAPES)
def test_argmax_rows(dtype, shape):
    rng = np.random.default_rng(shape[-1] + 1)
    x = P.round_bf16(rng.integers(-3, 4, shape).astype(np.float32))  # ties: the last position counts
    x.reshape(-1, shape[-1])[0, :shape[-1] // 2] = np.nan
    got, = run(lambda X: [Pop.argmax(X, len(shape) - 1)], [x], dtype, 'argmax')
    y = np.where(np.isnan(x), -np.inf, x)[..., ::-1]
    np.testing.assert_array_equal(got, shape[-1] - 1 - np.argmax(y, -1))


@pytest.mark.parametrize('dtype', ['f32', 'bf16', 'i32', 'u8'])
@pytest.mark.parametrize('direction', [P.SORT_ASC, P.SORT_DESC])
@pytest.mark.parametrize('rows,cols,k', [(1, 1, 1), (3, 10, 10), (5, 64, 3), (4, 65, 10), (9, 1000, 10), (6, 2561, 128), (2, 16384, 7)])
def test_first_of_a_sort(dtype, direction, rows, cols, k):
    rng = np.random.default_rng(cols + k)
    x = values(rng, (rows, cols), dtype)
    if dtype in ('f32', 'bf16'):
        x[:, ::3] = np.round(x[:, ::3])  # ties, zeros of both signs
        x[0, : cols // 4] = np.nan
    v, p = run(lambda X: list(Pop.topk(X, k, sort_direction=direction)), [x], dtype, 'top %d' % k)
    key = x.astype(np.float64)
    key = np.where(np.isnan(key), np.inf, -key if direction == P.SORT_DESC else key)
    want = np.argsort(key, 1, kind='stable')[:, :k]
    np.testing.assert_array_equal(p, want)
    np.testing.assert_array_equal(v.view(np.uint8), np.take_along_axis(x, want, 1).view(np.uint8))


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('shape', SHAPES + [(1030, 700), (3, 8192), (2, 8193)])
def test_softmax_rows(dtype, shape):
    rng = np.random.default_rng(shape[-1] + 2)
    x = values(rng, shape, dtype)
    got, = run(lambda X: [Pop.softmax(X, -1)], [x], dtype, 'softmax')
    e = np.exp(x.astype(np.float64) - x.max(-1, keepdims=True))
    want = e / e.sum(-1, keepdims=True)
    assert np.linalg.norm(got - want) < (1e-2 if dtype == 'bf16' else 2e-6) * np.linalg.norm(want)


@pytest.mark.parametrize('which', ['argmax', 'topk', 'softmax'])
def test_more_rows_than_one_launch_takes(which):
    """2^23 rows and some: they go in two launches, the second with the rows that are left."""
    rows, cols = (1 << 23) + 5, 3
    x = np.random.default_rng(9).random((rows, cols), dtype=np.float32)
    X = P.Placeholder(DT['f32'], x.shape)
    outs = {'argmax': lambda: [Pop.argmax(X, 1)], 'topk': lambda: list(Pop.topk(X, 2)), 'softmax': lambda: [Pop.softmax(X, 1)]}[which]()
    got = P.Runner(P.Program(which, [X], outs), target='hip').run([x])
    if which == 'argmax':
        np.testing.assert_array_equal(got[0], np.argmax(x, 1))  # (no ties among these)
    elif which == 'topk':
        order = np.argsort(-x, 1, kind='stable')[:, :2]
        np.testing.assert_array_equal(got[1], order)
        np.testing.assert_array_equal(got[0], np.take_along_axis(x, order, 1))
    else:
        e = np.exp(x - x.max(1, keepdims=True))
        np.testing.assert_allclose(got[0], e / e.sum(1, keepdims=True), rtol=2e-6)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('cols', [1, 31, 32, 33, 64, 65, 127, 128, 129])
@pytest.mark.parametrize('rows', [1, 7, 31, 33, 100])
def test_softmax_of_rows_that_share_a_wavefront(dtype, rows, cols):
    """Rows beside each other in one wavefront, the last ones missing: a row's maximum, sum, infinities and NaNs are its own."""
    rng = np.random.default_rng(rows * 1000 + cols)
    x = values(rng, (rows, cols), dtype) * 4
    if dtype == 'bf16':
        x = P.round_bf16(x)
    x[::5] += 64                            # (rows of another size; exact in bf16 up to rounding, rounded again below)
    if dtype == 'bf16':
        x = P.round_bf16(x)
    if cols > 1:
        x[::7, cols // 2] = -np.inf
    x[1::9, 0] = np.nan
    got, = run(lambda X: [Pop.softmax(X, -1)], [x], dtype, 'softmax')
    odd = np.isnan(x).any(1)
    assert np.isnan(got[odd]).all()
    e = np.exp(x[~odd].astype(np.float64) - x[~odd].max(-1, keepdims=True))
    want = e / e.sum(-1, keepdims=True)
    # (bf16: the difference, the exponential, the sum and the quotient rounded to 2^-9 each, the first of values up to 32)
    assert np.linalg.norm(got[~odd] - want) < (4e-2 if dtype == 'bf16' else 4e-6) * np.linalg.norm(want)

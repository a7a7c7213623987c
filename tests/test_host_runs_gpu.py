"""Runs on arrays in host memory (host/src/hip_runtime.cc, Runner) around the edges of their staging."""
import ctypes
import threading
import time

import numpy as np
import pytest
import torch

from plaidml_amd import edsl as P
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu
DT = {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16}


def test_an_allocation_that_fails_does_not_fail_the_next_launch():
    L = hk.lib()
    hk.init(0)
    ptr = ctypes.c_void_p()
    assert L.pml_hip_malloc(ctypes.byref(ptr), 1 << 50) != 0 and b'hipMalloc' in L.pml_hip_last_error()
    buf = hk.DeviceBuffer(4096)
    hk.check(L.pml_hip_fill_u32(buf.ptr, 0x01020304, 1024, None))
    np.testing.assert_array_equal(buf.to_numpy(np.uint32, (1024,)), 0x01020304)


def _program(dtype, n, m=300):
    X, Y = P.Placeholder(DT[dtype], [n]), P.Placeholder(DT[dtype], [m])
    return P.Program('host', [X, Y], [X * 2.0 + 1.0, Y - 1.0, X * -1.0])


def _round(a, dtype):
    return P.round_bf16(a) if dtype == 'bf16' else a


def _arrays(seed, dtype, n, m=300):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(n).astype(np.float32), rng.standard_normal(m).astype(np.float32)]


def _check(got, arrays, dtype):
    x, y = (_round(a, dtype) for a in arrays)
    # (rounded after each operation, as the separate operations round)
    want = [_round(_round(x * np.float32(2), dtype) + np.float32(1), dtype), _round(y - np.float32(1), dtype), -x]
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


# elements of a 4 MB piece, and of the 512 KB that still go by kernel
PIECE, KERNEL = {'f32': 1 << 20, 'bf16': 1 << 21}, {'f32': 1 << 17, 'bf16': 1 << 18}


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('pinned_results', [True, False])
@pytest.mark.parametrize('size', ['one', 'kernel', 'past kernel', 'piece', 'past piece', 'slots', 'past slots', 'two rounds'])
def test_arrays_around_the_sizes_of_the_staging(monkeypatch, dtype, pinned_results, size):
    """A value and its two results, with a small one beside them: copied by kernel, in a place of their own (32 MB in all),
    through the eight slots in turn; every run with other values."""
    k, p = KERNEL[dtype], PIECE[dtype]
    n = {'one': 1, 'kernel': k, 'past kernel': k + 1, 'piece': p, 'past piece': p + 1, 'slots': 8 * p // 3, 'past slots': 8 * p // 3 + 4096,
         'two rounds': 13 * p + 3}[size]
    if not pinned_results:
        monkeypatch.setattr(P, '_result_array', lambda dt, sizes, nbytes: np.empty(sizes, dt))
    runner = P.Runner(_program(dtype, n), target='hip')
    for run in range(4):
        arrays = _arrays(run, dtype, n)
        _check(runner.run(arrays), arrays, dtype)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
def test_runs_without_page_locked_memory(monkeypatch, dtype):
    """PLAIDML_PINNED=0 and a cap that is reached: ordinary copies; the staging is back as soon as there is memory for it."""
    n = PIECE[dtype] + 5
    runner = P.Runner(_program(dtype, n), target='hip')
    for run, (key, value) in enumerate([('PLAIDML_PINNED', '0'), ('PLAIDML_PINNED_MAX_MB', '1'), ('PLAIDML_PINNED', '1'), ('PLAIDML_PINNED_MAX_MB', '2')]):
        with monkeypatch.context() as patch:
            patch.setenv(key, value)
            arrays = _arrays(run, dtype, n)
            _check(runner.run(arrays), arrays, dtype)


@pytest.mark.parametrize('dtype,n', [('f32', 1000), ('bf16', 3 * PIECE['bf16'] + 1)])
def test_statistics_are_the_wall_time_in_three_parts(dtype, n):
    runner = P.Runner(_program(dtype, n), target='hip')
    for run in range(4):
        runner.run(_arrays(run, dtype, n))
        s = P.last_run_stats()
        assert s['kernel_ms'] > 0 and s['h2d_ms'] > 0 and s['d2h_ms'] >= 0
        # (the reading of the events themselves comes after the clock)
        assert s['h2d_ms'] + s['kernel_ms'] + s['d2h_ms'] == pytest.approx(runner.ms, rel=1e-6, abs=1e-9)


@pytest.mark.parametrize('n', [5, 70000, 600001])
def test_inputs_of_other_types_and_layouts(n):
    """bfloat16 as stored bits, arrays that are not contiguous, of another type, lists: what arrives is their value."""
    runner = P.Runner(_program('bf16', n), target='hip')
    x, y = _arrays(n, 'bf16', n)
    x[:3] = [np.nan, np.inf, -0.0]
    want = runner.run([x, y])
    _check([w[3:] if len(w) == n else w for w in want], [x[3:], y], 'bf16')
    wide = np.repeat(x, 2)
    for a in (P.to_bf16_bits(x), np.repeat(P.to_bf16_bits(x), 2)[::2], wide[::2], x.astype(np.float64), x[::-1].copy()[::-1], list(map(float, x)) if n < 10 else x):
        for g, w in zip(runner.run([a, y]), want):
            np.testing.assert_array_equal(g.view(np.uint32), w.view(np.uint32))


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
@pytest.mark.parametrize('n', [1000, 40000, 300000, 1200007])
def test_results_fed_back(dtype, n):
    """A result lies in page-locked memory and goes back from where it lies; so does a part of it that begins at any element."""
    X = P.Placeholder(DT[dtype], [n])
    runner = P.Runner(P.Program('step', [X], [X + 1.0]), target='hip')
    x = np.arange(n, dtype=np.float32) % 100
    first, = runner.run([x])
    second, = runner.run([first])
    np.testing.assert_array_equal(first, x + 1)  # (the second run left the first one's results alone)
    np.testing.assert_array_equal(second, x + 2)
    Y = P.Placeholder(DT[dtype], [n - 3])
    part = P.Runner(P.Program('step', [Y], [Y + 1.0]), target='hip')
    for _ in range(4):
        got, = part.run([second[1:n - 2]])
        np.testing.assert_array_equal(got, x[1:n - 2] + 3)
        got, = part.run([second[::-1][:n - 3]])
        np.testing.assert_array_equal(got, x[::-1][:n - 3] + 3)


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
def test_runs_from_several_threads(dtype):
    """An executable of its own per thread; their passes over arrays share the helper threads, which only one of them gets."""
    n, wrong = 3 * PIECE[dtype] + 11, []

    def work(seed):
        try:
            runner = P.Runner(_program(dtype, n), target='hip')
            for run in range(4):
                arrays = _arrays(10 * seed + run, dtype, n)
                _check(runner.run(arrays), arrays, dtype)
                assert runner.ms > 0
        except BaseException as e:  # noqa: B902
            wrong.append(e)
    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[0]


@pytest.mark.parametrize('dtype', ['f32', 'bf16'])
def test_outputs_hold_the_last_run_of_either_kind(dtype):
    n = 50000
    runner = P.Runner(_program(dtype, n), target='hip')
    sets = [_arrays(s, dtype, n) for s in range(4)]
    staged = runner.stage(sets[1])
    _check(runner.run(sets[0]), sets[0], dtype)
    _check(runner.fetch(), sets[0], dtype)
    runner.run_staged(staged)
    _check(runner.fetch(), sets[1], dtype)
    kept = runner.run(sets[2])
    _check(runner.fetch(), sets[2], dtype)
    _check(runner.run(sets[3]), sets[3], dtype)
    _check(kept, sets[2], dtype)
    runner.run_staged(staged)
    _check(runner.fetch(), sets[1], dtype)


def test_arrays_that_do_not_fit_are_refused():
    runner = P.Runner(_program('f32', 100), target='hip')
    x, y = _arrays(0, 'f32', 100)
    with pytest.raises(Exception):
        runner.run([x[:99], y])
    with pytest.raises(Exception):
        runner.run([x])
    _check(runner.run([x, y]), [x, y], 'f32')


@pytest.mark.parametrize('layers', [1, 4, 10])
def test_a_call_leaves_nothing_to_whoever_waits_next(layers):
    """A call on host arrays returns when its stream is through: waiting for the device behind it takes what it takes again at once."""
    rng = np.random.default_rng(layers)
    X = P.Placeholder(P.DType.FLOAT32, [20, 64])
    x, i, j, k = X, *P.TensorIndexes(3)
    for _ in range(layers):
        W = P.Constant(rng.standard_normal((64, 64)).astype(np.float32) / 8, P.DType.FLOAT32)
        x = P.Contraction().outShape(20, 64).outAccess(i, j).sum(x[i, k] * W[k, j]).build()
    runner = P.Runner(P.Program('layers', [X], [x]), target='hip')
    arrays = [rng.standard_normal((20, 64)).astype(np.float32)]
    behind, again = [], []
    for _ in range(210):
        runner.run(arrays)
        t = [time.perf_counter()]
        for _ in range(2):
            torch.cuda.synchronize()
            t.append(time.perf_counter())
        behind.append(t[1] - t[0])
        again.append(t[2] - t[1])
    first, second = sorted(behind[10:])[100], sorted(again[10:])[100]
    print('%d layers: %.1f us behind a call, %.1f again' % (layers, first * 1e6, second * 1e6), flush=True)
    assert first < 2 * second + 2e-6

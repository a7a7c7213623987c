"""The host side of a run that makes no GPU calls (host/src/host_copy.cc, pinned_pool.cc), compiled by itself: rounding to and
from bfloat16 against numpy, lengths around where helper threads join, several threads at once, and the pool's limits."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, 'plaidml_amd', 'host', 'src')
FILES = [os.path.join(ROOT, 'tests', 'cpp', 'host_memory.cc'), os.path.join(SRC, 'host_copy.cc'), os.path.join(SRC, 'pinned_pool.cc')]
PIECE = 65536  # fp32 values of a piece; up to two pieces stay with the caller's thread


def _build(out, *flags):
    subprocess.check_call(['g++', '-std=c++17', '-O3', '-I' + SRC, *flags, *FILES, '-pthread', '-o', str(out)])
    return str(out)


@pytest.fixture(scope='module')
def lib(tmp_path_factory):
    L = ctypes.CDLL(_build(tmp_path_factory.mktemp('host') / 'libhost.so', '-shared', '-fPIC'))
    vp, sz = ctypes.c_void_p, ctypes.c_size_t
    for name in ('to_bf16', 'from_bf16', 'copy'):
        getattr(L, name).argtypes, getattr(L, name).restype = [vp, vp, sz], None
    for name, args, res in (('pool_new', [sz, sz], vp), ('pool_take', [vp, sz, sz], vp), ('pool_put', [vp, vp], None),
                            ('pool_holds', [vp, vp, sz], ctypes.c_int), ('pool_total', [vp], sz), ('system_given', [], sz), ('system_most', [], sz)):
        getattr(L, name).argtypes, getattr(L, name).restype = args, res
    return L


def _rounded(x):
    """Round to nearest even in integer arithmetic; any NaN 0x7fc0."""
    u = x.view(np.uint32).astype(np.uint64)
    r = ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return np.where(np.isnan(x), np.uint16(0x7fc0), r)


SPECIAL = np.array([0x00000000, 0x80000000, 0x7f800000, 0xff800000, 0x7fc00000, 0x7f800001, 0xffffffff, 0x7f80ffff, 0x7f7fffff, 0xff7fffff,
                    0x3f808000, 0x3f818000, 0x3f808001, 0x3f807fff, 0x00000001, 0x00008000, 0x00018000, 0x807fffff, 0x7f7f8000, 0x7f7f7fff],
                   np.uint32).view(np.float32)  # zeros, infinities, NaNs of several payloads, ties to even, denormals, the edge of overflow


@pytest.mark.parametrize('n', [0, 1, 7, 15, 33, 2 * PIECE - 1, 2 * PIECE, 2 * PIECE + 1, 3 * PIECE + 5, 17 * PIECE + 3])
def test_rounding_to_and_from_bfloat16(lib, n):
    x = np.random.default_rng(n).integers(0, 1 << 32, n + 8, dtype=np.uint64).astype(np.uint32).view(np.float32)
    at = np.random.default_rng(1).integers(0, max(n, 1), min(n, 200))
    x[at] = SPECIAL[np.arange(len(at)) % len(SPECIAL)]
    if n:
        x[n - 1] = SPECIAL[5]
    for shift in (0, 1):  # (a start that is no whole vector)
        src, bits, back = x[shift:shift + n].copy(), np.full(n + 2, 0xabcd, np.uint16), np.full(n + 2, 7, np.float32)
        lib.to_bf16(bits[1:].ctypes.data, src.ctypes.data, n)
        np.testing.assert_array_equal(bits[1:n + 1], _rounded(src))
        assert bits[0] == 0xabcd and bits[n + 1] == 0xabcd
        lib.from_bf16(back[1:].ctypes.data, bits[1:].ctypes.data, n)
        np.testing.assert_array_equal(back[1:n + 1].view(np.uint32), bits[1:n + 1].astype(np.uint32) << 16)
        assert back[0] == 7 and back[n + 1] == 7


@pytest.mark.parametrize('n', [0, 1, 4 * PIECE - 1, 8 * PIECE, 8 * PIECE + 1, 40 * PIECE + 11])
def test_copies(lib, n):
    src = np.random.default_rng(n).integers(0, 256, n + 1, dtype=np.uint8)
    dst = np.zeros(n + 3, np.uint8)
    lib.copy(dst[1:].ctypes.data, src[1:].ctypes.data, n)
    np.testing.assert_array_equal(dst[1:n + 1], src[1:])
    assert dst[0] == 0 and dst[n + 1] == 0


@pytest.mark.parametrize('sanitizer', ['thread', 'address,undefined'])
def test_long_passes_from_several_threads(tmp_path, sanitizer):
    # (the loops' variants per processor are chosen before a sanitizer's runtime is up: without them here)
    exe = _build(tmp_path / 'passes', '-g', '-fsanitize=' + sanitizer, '-Dtarget_clones(...)=')
    subprocess.run([exe], check=True, timeout=300)


MB = 1 << 20


def test_pool_counts_what_it_keeps_and_what_it_rounds_up(lib):
    pool = lib.pool_new(256 * MB, 1 << 40)
    cap = 10 * MB
    a, b = lib.pool_take(pool, 4 * MB, cap), lib.pool_take(pool, 4 * MB, cap)
    assert a and b and lib.pool_total(pool) == 8 * MB == lib.system_given()
    assert not lib.pool_take(pool, 4 * MB, cap)
    lib.pool_put(pool, a)
    lib.pool_put(pool, b)
    assert lib.pool_total(pool) == 8 * MB            # kept for the next one of their size ...
    assert lib.pool_take(pool, 4 * MB, cap) == b     # (the one freed last)
    c = lib.pool_take(pool, 5 * MB, cap)             # ... and given back for one that needs the room
    assert c and lib.pool_total(pool) == 9 * MB == lib.system_given()
    assert lib.system_most() <= cap
    lib.pool_put(pool, b)
    lib.pool_put(pool, c)
    # 4.1 MB take 4.5: three are 13.5 and not 12.3
    big = [lib.pool_take(pool, int(4.1 * MB), 13 * MB) for _ in range(3)]
    assert big[0] and big[1] and not big[2] and lib.system_most() <= 13 * MB
    for p in big[:2]:
        lib.pool_put(pool, p)
    assert lib.pool_take(pool, int(12.9 * MB), int(13 * MB)) and lib.system_given() <= 13 * MB  # (up to the cap itself)


def test_pool_gives_back_what_it_keeps_when_the_system_has_no_more(lib):
    pool = lib.pool_new(256 * MB, 12 * MB)
    a = lib.pool_take(pool, 8 * MB, 1 << 40)
    assert not lib.pool_take(pool, 6 * MB, 1 << 40)  # in use: nothing to be had ...
    assert lib.pool_total(pool) == 8 * MB            # ... and nothing left booked
    lib.pool_put(pool, a)
    assert lib.pool_take(pool, 6 * MB, 1 << 40)      # kept: given back for it
    assert lib.system_given() == 6 * MB == lib.pool_total(pool)


def test_pool_keeps_within_its_bound_and_knows_its_blocks(lib):
    pool = lib.pool_new(8 * MB, 1 << 40)
    blocks = [lib.pool_take(pool, 3 * MB, 1 << 40) for _ in range(4)]
    assert lib.pool_holds(pool, blocks[1], 3 * MB) and lib.pool_holds(pool, blocks[1] + MB, 2 * MB)
    assert not lib.pool_holds(pool, blocks[1] + MB, 3 * MB) and not lib.pool_holds(pool, 4096, 1)
    for p in blocks:
        lib.pool_put(pool, p)
    assert lib.pool_total(pool) == 6 * MB == lib.system_given()
    assert not lib.pool_holds(pool, blocks[3], 1)    # kept ones are nobody's
    lib.pool_put(pool, blocks[3])                    # (a second time: no block in use)
    lib.pool_put(pool, None)
    assert lib.pool_total(pool) == 6 * MB
    assert lib.pool_take(pool, 0, 1 << 40) and not lib.pool_take(pool, 2 * MB, MB)

"""Copies between host arrays and states through pinned staging memory (marked gpu): pieces of 1 MiB on four slots,
threads from 8 MiB on. Every byte has to arrive, at sizes around those of a piece, the slots and a
thread's share, and from several threads at once."""
import ctypes
import threading

import numpy
import pytest

from qip_amd import GpuBackend
from qip_amd.batch import GpuBatch

pytestmark = pytest.mark.gpu
MIB = 2 ** 17                     # complex64 amplitudes in 1 MiB


def vector(count, seed, dtype=numpy.complex64):
    rng = numpy.random.default_rng(seed)
    return (rng.standard_normal(count) + 1j * rng.standard_normal(count)).astype(dtype)


@pytest.mark.parametrize("start,count", [(0, 1), (5, 3), (1, MIB - 1), (0, MIB), (7, MIB + 1), (0, 4 * MIB), (3, 4 * MIB + 5),
                                         (0, 5 * MIB), (1, 8 * MIB - 1), (0, 8 * MIB), (9, 12 * MIB + 3), (0, 16 * MIB),
                                         (11, 19 * MIB + 77), (0, 32 * MIB)])
def test_ranges_arrive_whole(start, count):
    be = GpuBackend.make_state(22, [], [], statetype=numpy.complex64)
    v = vector(count, count)
    be.overwrite_relative_range(start, start + count, v)
    assert numpy.array_equal(be.get_relative_range(start, start + count), v)
    rest = be.get_state()
    assert numpy.array_equal(rest[start:start + count], v)
    rest[start:start + count] = 0
    rest[0] = 0
    assert not rest.any()
    be.addto_relative_range(start, start + count, v)
    assert numpy.array_equal(be.get_relative_range(start, start + count), v + v)
    be.close()


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n", [1, 2, 5, 12, 21])
def test_basis_state(n, dtype):
    be = GpuBackend.make_state(n, [], [], statetype=dtype)
    be.kronselect_dot({n - 1: numpy.array([[0.0, 1.0], [1.0, 0.0]])})
    be.reinit()
    want = numpy.zeros(2 ** n, dtype=dtype)
    want[0] = 1
    assert numpy.array_equal(be.get_state(), want)
    be.close()


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("kinds", [("f8", "c16"), ("f4", "i8"), ("c8", "f8"), ("?", "f8")])
@pytest.mark.parametrize("lens", [(1, 3), (18, 3), (2, 19)])
def test_real_feeds_equal_complex_ones(lens, kinds, dtype):
    rng = numpy.random.default_rng(sum(lens))
    n = sum(lens)
    perm = [int(q) for q in rng.permutation(n)]
    groups = [perm[:lens[0]], perm[lens[0]:]]
    feeds = [(rng.standard_normal(2 ** k) * 3).astype(kind) for k, kind in zip(lens, kinds)]
    a = GpuBackend.make_state(n, groups, feeds, statetype=dtype)
    b = GpuBackend.make_state(n, groups, [f.astype(numpy.complex128) for f in feeds], statetype=dtype)
    assert numpy.array_equal(a.get_state(), b.get_state())
    a.reinit([list(range(n))], [numpy.arange(2 ** n)])
    assert numpy.array_equal(a.get_state(), numpy.arange(2 ** n).astype(dtype))
    a.close()
    b.close()


@pytest.mark.parametrize("start,count", [(0, 479), (1, 480), (2, 481), (3, 482), (1, 16384), (1, 16385)])
def test_short_ranges_arrive_whole(start, count):
    test_ranges_arrive_whole(start, count)      # around what travels as kernel arguments, and 128 KiB


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("kinds", [("f8", "c16"), ("f4", "i8"), ("c8", "f8"), ("?", "f8")])
@pytest.mark.parametrize("lens", [(12, 1), (13, 2), (11, 13)])
def test_real_feeds_around_the_short_ones_equal_complex_ones(lens, kinds, dtype):
    test_real_feeds_equal_complex_ones(lens, kinds, dtype)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("lens", [(13, 1, 1), (1, 14, 2), (12, 1, 7), (2, 12, 4), (1,) * 15, (3, 2, 13)])
def test_feeds_short_and_long_are_the_product_of_their_groups(lens, dtype):
    rng = numpy.random.default_rng(len(lens) + sum(lens))
    n = sum(lens)
    perm = [int(q) for q in rng.permutation(n)]
    groups, feeds, at = [], [], 0
    for k in lens:
        groups.append(perm[at:at + k])
        feeds.append(rng.standard_normal(2 ** k) + (0 if at % 2 else 1j * rng.standard_normal(2 ** k)))
        at += k
    want = numpy.ones(2 ** n, dtype=numpy.complex128)
    i = numpy.arange(2 ** n)
    for g, f in zip(groups, feeds):
        value = numpy.zeros(2 ** n, dtype=numpy.int64)
        for q in g:
            value = value << 1 | (i >> (n - 1 - q) & 1)
        want *= f[value]
    be = GpuBackend.make_state(n, groups, feeds, statetype=dtype)
    eps = numpy.finfo(dtype).eps
    # a rounding per product, and one on the way to the state's precision
    assert numpy.max(numpy.abs(be.get_state() - want) / numpy.abs(want)) < 4 * len(lens) * 2.3e-16 + 2 * eps
    be.close()


def test_feeds_beyond_the_groups_are_left_out():
    one, zero = numpy.array([0.0, 1.0]), numpy.array([1.0, 0.0])
    for groups, feeds, at in (([], [one], 0), ([[0]], [one, zero], 4), ([[2], [0]], [one, one, numpy.ones(2 ** 14)], 5)):
        be = GpuBackend.make_state(3, groups, feeds)
        assert numpy.array_equal(be.get_state(), numpy.arange(8) == at)
        be.close()


def test_a_real_feed_takes_no_more_device_memory_than_a_complex_one():
    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n, used, states = 25, [], []
    for dtype in (numpy.float64, numpy.complex128, numpy.float64):      # the first use of a kernel takes memory too
        feed = numpy.zeros(2 ** n, dtype=dtype)
        feed[12345] = 1.0
        free = free_bytes()
        be = GpuBackend.make_state(n, [list(range(n))[::-1]], [feed])
        be.synchronize()
        used.append(free - free_bytes())
        at = int(format(12345, '025b')[::-1], 2)
        assert be.get_relative_range(at, at + 1)[0] == 1.0 and be.total_prob() == 1.0
        states.append(be)
    print("device memory of a state with a real, a complex and a real feed", used, flush=True)
    for be in states:
        be.close()
    assert used[2] <= used[1] + (16 << 20)


def test_threads_read_and_write_their_own_states():
    n, wrong = 20, []

    def work(seed):
        be = GpuBackend.make_state(n, [], [])
        for i in range(3):
            v = vector(2 ** n, 10 * seed + i, numpy.complex128)
            be.overwrite_relative_range(0, 2 ** n, v)
            if not numpy.array_equal(be.get_state(), v):
                wrong.append((seed, i))
        be.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(10)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_batch_states():
    ns = [3, 17, 18, 20, 21]
    b = GpuBatch(ns)
    vs = [vector(2 ** n, n) for n in ns]
    for i, v in enumerate(vs):
        b.set_state(i, v)
    for i, v in enumerate(vs):
        assert numpy.array_equal(b.get_state(i), v)
    b.close()

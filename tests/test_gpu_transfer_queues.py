"""Copies of one state while another has work queued (marked gpu): a copy waits for its own state's queue only. "Still
busy" is told by the time that the other state's synchronize takes afterwards."""
import time

import numpy
import pytest

from qip_amd import GpuBackend
from qip_amd.batch import GpuBatch

pytestmark = pytest.mark.gpu


def vector(count, seed, dtype=numpy.complex64):
    rng = numpy.random.default_rng(seed)
    return (rng.standard_normal(count) + 1j * rng.standard_normal(count)).astype(dtype)


def busy_state(seconds=0.6):
    """A state and a function that queues about `seconds` of work on it, by sweeps timed on the spot."""
    a = GpuBackend.make_state(28, [], [])
    rng = numpy.random.default_rng(1)
    u = numpy.linalg.qr(rng.standard_normal((8, 8)) + 1j * rng.standard_normal((8, 8)))[0]

    def sweeps(count):
        for _ in range(count):
            a.kronselect_dot({(0, 9, 18): u})
        a.flush()

    sweeps(5)
    a.synchronize()
    t = time.perf_counter()
    sweeps(20)
    a.synchronize()
    each = (time.perf_counter() - t) / 20
    return a, lambda: sweeps(max(1, int(seconds / each)))


def returns_first(a, work, calls):
    """Whether any of the calls, each after fresh work on `a`, returns well before that work is done. (Several, because
    two streams may share one of the card's hardware queues, where the second does wait.)"""
    for i, call in enumerate(calls):
        work()
        print("queued, call", i, flush=True)
        call()
        t = time.perf_counter()
        a.synchronize()
        if time.perf_counter() - t > 0.1:
            return True
    return False


@pytest.mark.parametrize("what", ["read", "read 8 MiB", "write", "init", "batch"])
def test_a_copy_does_not_wait_for_another_states_queue(what):
    a, work = busy_state()
    up = vector(5, 2, numpy.complex128)
    others = [GpuBackend.make_state(19, [], []) for _ in range(5)]
    batch = GpuBatch([10, 11]) if what == "batch" else None
    v = vector(2 ** 19, 3, numpy.complex128)
    for b in others:
        b.overwrite_relative_range(0, 2 ** 19, v)
        assert numpy.array_equal(b.get_state(), v)

    def call(b):
        a.overwrite_relative_range(1, 6, up)        # an upload behind the work
        if what == "read":
            assert numpy.array_equal(b.get_relative_range(3, 9), v[3:9])
        elif what == "read 8 MiB":
            assert numpy.array_equal(b.get_state(), v)
        elif what == "write":
            b.overwrite_relative_range(0, 4, v[:4])
            b.synchronize()
        elif what == "init":
            b.reinit([[0, 1], [2]], [numpy.array([1.0, 0, 0, 0]), numpy.array([0.0, 1.0])])
            b.synchronize()
        else:
            batch.set_state(1, v[:2 ** 11].astype(numpy.complex64))
            assert numpy.array_equal(batch.get_state(1), v[:2 ** 11].astype(numpy.complex64))

    assert returns_first(a, work, [lambda b=b: call(b) for b in others])
    assert numpy.array_equal(a.get_relative_range(1, 6), up)
    for b in others + [a] + ([batch] if batch else []):
        b.close()


def test_fed_initialisations_do_not_wait_for_their_own_queue():
    """Ten of them behind queued work: each is one copy, and all of them return before the work is done."""
    a, work = busy_state()
    rng = numpy.random.default_rng(4)
    feeds = [rng.standard_normal(2) + (0 if q % 2 else 1j * rng.standard_normal(2)) for q in range(28)]
    feeds = [f / numpy.linalg.norm(f) for f in feeds]
    groups = [[q] for q in range(28)]
    work()
    for _ in range(10):
        a.reinit(groups, feeds)
    t = time.perf_counter()
    a.synchronize()
    assert time.perf_counter() - t > 0.1
    want = numpy.ones(1, dtype=numpy.complex128)
    for f in feeds[14:]:
        want = numpy.kron(want, f)
    lead = numpy.prod([f[0] for f in feeds[:14]])
    assert numpy.max(numpy.abs(a.get_relative_range(0, 2 ** 14) - lead * want)) < 1e-15
    a.close()


def test_more_uploads_behind_one_queue_than_there_is_staging_memory():
    a, work = busy_state(0.3)
    work()
    vs = [vector(2 ** 16 if i % 8 == 0 else 11 + i, i, numpy.complex128) for i in range(45)]
    for i, v in enumerate(vs):
        a.overwrite_relative_range(i << 17, (i << 17) + len(v), v)
    b = GpuBackend.make_state(20, [], [])
    w = vector(2 ** 20, 99, numpy.complex128)
    b.overwrite_relative_range(0, 2 ** 20, w)
    assert numpy.array_equal(b.get_state(), w)
    for i, v in enumerate(vs):
        assert numpy.array_equal(a.get_relative_range(i << 17, (i << 17) + len(v)), v)
    a.close()
    b.close()

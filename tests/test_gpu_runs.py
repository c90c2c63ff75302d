"""Held-back runs (marked gpu): single-qubit gates, swaps and diagonals under any controls wait on the
state and go in passes over 4096-amplitude tiles, gates that round nothing (X, swaps, -1 factors)
joining an earlier pass where that changes no value. Every run must equal, bit for bit, the same gates
each launched alone (a synchronisation after every gate), and be within 1e-12 of the oracle."""
import numpy
import pytest

from oracle.oracle_backend import OracleBackend
from qip_amd import CMat, GpuBackend, SwapMat
from qip_amd.backend import max_abs_diff

pytestmark = pytest.mark.gpu
HM = numpy.array([[1.0, 1.0], [1.0, -1.0]]) / numpy.sqrt(2.0)
XM = numpy.array([[0.0, 1.0], [1.0, 0.0]])
ZM = numpy.diag([1.0, -1.0])


def unitary(rng):
    z = rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2))
    q, r = numpy.linalg.qr(z)
    return q * (numpy.diagonal(r) / numpy.abs(numpy.diagonal(r)))


def gate(rng, n):
    """A held gate on random qubits: Haar, H, X, phases, Z, a two-target diagonal or a swap, under up to
    three controls."""
    kind = int(rng.integers(0, 8))
    width = 2 if kind in (5, 6) and n >= 2 else 1
    controls = int(min(rng.integers(0, 4), n - width)) if rng.random() < 0.6 else 0
    qs = tuple(int(q) for q in rng.permutation(n)[:controls + width])
    if width == 2:
        m = SwapMat(1) if kind == 5 else numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 4)))
    else:
        m = [unitary(rng), HM, XM, ZM, numpy.diag([1.0, numpy.exp(1j * rng.uniform(0, 6))]),
             numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 2))), XM, unitary(rng)][kind]
    for _ in range(controls):
        m = CMat(m)
    return {qs: m}


def check(n, dtype, seq, rng, oracle):
    psi = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
    psi /= numpy.linalg.norm(psi)
    held = GpuBackend.make_state(n, [list(range(n))], [psi], statetype=dtype)
    alone = GpuBackend.make_state(n, [list(range(n))], [psi], statetype=dtype)
    for d in seq:
        held.kronselect_dot(d)
        alone.kronselect_dot(d)
        alone.synchronize()
    got = held.get_state()
    assert numpy.array_equal(got, alone.get_state())
    if oracle:
        ora = OracleBackend.make_state(n, [list(range(n))], [psi])
        for d in seq:
            ora.kronselect_dot(d)
        assert numpy.max(numpy.abs(got - ora.get_state())) < 1e-12
    held.close()
    alone.close()


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 11, 12, 13, 17, 22])
def test_mixed_runs_equal_separate_launches(n, dtype):
    rng = numpy.random.default_rng(700 + n)
    print("mixed runs n", n, numpy.dtype(dtype).name, flush=True)
    check(n, dtype, [gate(rng, n) for _ in range(230)], rng, dtype == numpy.complex128 and n <= 13)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("low", [False, True])
def test_layers_whose_two_qubit_gates_straddle_tiles(low, dtype):
    """Haar layers with CNOTs, swaps and CZs between neighbours and across the register: the two-qubit
    gates join passes whose tiles hold only the bits they change; targets on every tile position."""
    n = 21
    rng = numpy.random.default_rng(31 + low)
    seq = []
    for layer in range(5):
        qs = list(range(n))[::-1 if low else 1]
        seq += [{q: unitary(rng)} for q in qs]
        seq += [{(q, q + 1): CMat(XM if layer % 2 else ZM)} for q in range(layer % 2, n - 1, 2)]
        seq += [{(q, n - 1 - q): SwapMat(1)} for q in range(layer, n // 2, 2)]
        seq += [{(n - 1 - q, q): CMat(numpy.diag([1.0, numpy.exp(0.3j * q)]))} for q in range(n // 2)]
    print("layers n", n, numpy.dtype(dtype).name, "low" if low else "high", flush=True)
    check(n, dtype, seq, rng, False)


def test_runs_longer_than_a_launch_holds():
    """More diagonals and coefficients than one launch's arguments hold, between gates that change bits."""
    n = 14
    rng = numpy.random.default_rng(5)
    seq = []
    for t in range(n):
        seq.append({t: HM})
        seq += [{(i, t): CMat(numpy.diag([1.0, numpy.exp(2j * numpy.pi / 2 ** (1 + i - t))]))} for i in range(t + 1, n)]
    seq += [{(i, n - 1 - i): SwapMat(1)} for i in range(n // 2)]
    seq += [{(0, 1): numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 4)))} for _ in range(70)]
    check(n, numpy.complex128, seq, rng, True)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n", [4, 9, 10, 14, 19, 20])
def test_every_target_and_control_of_small_states(n, dtype):
    """Every operation kind on every target, with the control just above and just below it, on states of
    one tile of 1024, of several, and on either side of the size at which tiles become 4096."""
    rng = numpy.random.default_rng(90 + n)
    seq = []
    for t in range(n):
        above, below = (t + 1) % n, (t - 1) % n
        seq += [{t: unitary(rng)}, {t: HM}, {(above, t): CMat(XM)}, {(below, t): CMat(unitary(rng))}, {t: XM},
                {(above, t): CMat(numpy.diag([1.0, numpy.exp(0.7j)]))}, {(t, below): CMat(ZM)},
                {(t, (t + n // 2) % n): SwapMat(1)}, {(below, t): numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 4)))}]
    print("targets n", n, numpy.dtype(dtype).name, flush=True)
    check(n, dtype, seq, rng, dtype == numpy.complex128 and n <= 10)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n", [11, 13, 16, 20, 22])
def test_swaps_that_move_together(n, dtype):
    """Swaps in one exchange: a register's reversal, its halves, swaps that share bits, swaps behind and
    before gates on their bits, under a control and on the lowest bits."""
    rng = numpy.random.default_rng(17 + n)
    sw = lambda a, b: {(a, b): SwapMat(1)}    # noqa: E731
    seq = [sw(i, n - 1 - i) for i in range(n // 2)]
    seq += [{0: unitary(rng)}, {n - 1: HM}] + [sw(i, i + n // 2) for i in range(n // 2)]
    seq += [sw(0, 1), sw(1, 2), sw(2, 0), {1: unitary(rng)}, sw(3, 1), {(0, 3, 5): CMat(SwapMat(1))}, sw(5, 6)]
    seq += [{(2, 4): CMat(XM)}, sw(2, 3), sw(4, n - 1), {4: HM}, {(n - 2, n - 3): numpy.diag([1, 1j, -1, 1.0])}, sw(n - 2, 0)]
    print("swaps n", n, numpy.dtype(dtype).name, flush=True)
    check(n, dtype, seq, rng, dtype == numpy.complex128 and n <= 13)


@pytest.mark.parametrize("n,dtype", [(25, numpy.complex128), (26, numpy.complex128), (26, numpy.complex64), (27, numpy.complex64)])
def test_a_swap_alone_on_either_side_of_the_caches(n, dtype):
    """512 MiB and 1 GiB: swaps each by itself against the same ones together."""
    rng = numpy.random.default_rng(n)
    groups = [list(range(0, n, 2)), list(range(1, n, 2))]
    feeds = [rng.standard_normal(2 ** len(g)) + 1j * rng.standard_normal(2 ** len(g)) for g in groups]
    states = [GpuBackend.make_state(n, groups, feeds, statetype=dtype) for _ in range(2)]
    swaps = [(0, 1), (2, n - 5), (n // 2, 5)]
    for a, b in swaps:
        states[0].kronselect_dot({(a, b): SwapMat(1)})
        states[1].kronselect_dot({(a, b): SwapMat(1)})
        states[1].synchronize()
    assert max_abs_diff(*states) == 0.0
    for a, b in swaps[::-1]:
        states[0].kronselect_dot({(b, a): SwapMat(1)})
        states[0].flush()
    states[1].reinit(groups, feeds)
    assert max_abs_diff(*states) == 0.0
    for s in states:
        s.close()


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n", [18, 19, 20])
def test_layers_of_single_qubit_operators_around_the_size_where_tiles_change(n, dtype):
    """Layers of nothing else (on 19 qubits tiles of 4096), with a phase at the end of one (tiles of 1024), and between
    gates under controls."""
    rng = numpy.random.default_rng(1900 + n)
    layer = lambda m: [{int(q): m()} for q in rng.permutation(n)]    # noqa: E731
    seq = layer(lambda: unitary(rng)) + layer(lambda: HM) + layer(lambda: XM)
    seq += [{3: numpy.diag([1.0, 1j])}] + layer(lambda: unitary(rng)) + [{(n - 1, 4): CMat(XM)}] + layer(lambda: XM) * 5
    check(n, dtype, seq, rng, False)

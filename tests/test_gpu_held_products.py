"""Products of single-qubit operators held back on the state (marked gpu): products that follow each other are
multiplied, and two products around diagonals share a pass; against the factors applied one by one in
numpy, in complex128."""
import numpy
import pytest

from qip_amd import CMat, GpuBackend
from qip_amd.fused import FusedBackend

pytestmark = pytest.mark.gpu
HM = numpy.array([[1.0, 1.0], [1.0, -1.0]]) / numpy.sqrt(2.0)
XM = numpy.array([[0.0, 1.0], [1.0, 0.0]])


def unitary(rng):
    z = rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2))
    q, r = numpy.linalg.qr(z)
    return q * (numpy.diagonal(r) / numpy.abs(numpy.diagonal(r)))


def controlled(m, levels):
    for _ in range(levels):
        m = CMat(m)
    return m


def apply(psi, n, d):
    """A descriptor of single-qubit factors, or one matrix under controls, on the amplitudes psi."""
    v = psi.reshape((2,) * n)
    for key, m in d.items():
        key, ctl = (key,) if isinstance(key, int) else key, 0
        while isinstance(m, CMat):
            m, ctl = m.m, ctl + 1
        k = len(key) - ctl
        v = v.copy()
        on = [slice(None)] * n
        for q in key[:ctl]:
            on[q] = 1
        sub = v[tuple(on)]                       # its axes are the qubits that are not controls
        axes = [q - sum(c < q for c in key[:ctl]) for q in key[ctl:]]
        out = numpy.tensordot(numpy.asarray(m).reshape((2,) * (2 * k)), sub, axes=(list(range(k, 2 * k)), axes))
        v[tuple(on)] = numpy.moveaxis(out, list(range(k)), axes)
    return v.reshape(-1)


def layer(bits, n, f):
    return {n - 1 - b: f() for b in bits}


def diagonals(n, bits, kind, rng):
    """Diagonals between two products: none; a phase under every bit of the products; one under a control
    in each part of the state; two targets; or more than may stand between two held products."""
    q = [n - 1 - b for b in bits]
    phase = numpy.diag([1.0, numpy.exp(1.3j)])
    if kind == "none":
        return []
    if kind == "all":
        return [{tuple(q): controlled(numpy.diag([1.0, -1.0]), len(q) - 1)}]
    if kind == "some":
        return [{(q[0], q[-1]): CMat(phase)}, {(0, n - 1): CMat(phase)}, {(q[-1],): numpy.diag(numpy.exp([1j, 2j]))}]
    if kind == "two":
        return [{(q[-1], q[0]): numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 4)))},
                {(1, q[-1], q[1]): CMat(numpy.diag(numpy.exp(1j * rng.uniform(0, 6, 4))))}]
    return [{(a, b): CMat(phase)} for a, b in zip(range(0, 6), range(6, 12))]


def check(make, n, seq, rng, dtype, tol):
    psi = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
    psi /= numpy.linalg.norm(psi)
    be = make(n, [list(range(n))], [psi], statetype=dtype)
    ref = psi
    for d in seq:
        be.kronselect_dot(d)
        ref = apply(ref, n, d)
    assert numpy.max(numpy.abs(be.get_state() - ref)) < tol * 2 ** (-n / 2) * 50
    be.close()


# a recording backend composes narrow diagonals into blocks of its own: with it, diagonals wider than those
@pytest.mark.parametrize("make,dtype,tol,between", [
    (GpuBackend.make_state, dtype, tol, between) for dtype, tol in ((numpy.complex128, 1e-13), (numpy.complex64, 1e-6))
    for between in ("none", "all", "some", "two", "many")] + [(FusedBackend.make_state, numpy.complex64, 1e-6, "all")])
@pytest.mark.parametrize("n,bits", [
    (12, range(12)),                  # one pass takes every bit
    (14, range(4, 12)),               # eight high bits, all in the shared pass
    (14, range(6, 14)),
    (13, range(13)),                  # one high bit left for the shared pass
    (16, range(1, 16)),               # four: no move through LDS
    (17, range(17)),                  # five: the first on a bit that needs one
    (20, range(20)),                  # eight
    (18, [1, 4, 6, 9, 10, 11, 12, 13, 14, 15, 16, 17]),
])
def test_products_around_diagonals(n, bits, make, dtype, tol, between):
    rng = numpy.random.default_rng(n + len(between))
    print("held products", n, list(bits), between, numpy.dtype(dtype).name, make.__self__.__name__, flush=True)
    u = lambda: unitary(rng)    # noqa: E731
    h, x = (lambda: HM), (lambda: XM)
    for first, second in (((u,), (u,)), ((h, x), (x, h)), ((x,), (x,))):
        seq = [layer(bits, n, f) for f in first] + diagonals(n, list(bits), between, rng)
        check(make, n, seq + [layer(bits, n, f) for f in second], rng, dtype, tol)


@pytest.mark.parametrize("dtype,tol", [(numpy.complex128, 1e-13), (numpy.complex64, 1e-6)])
def test_products_of_unlike_bits_and_kinds(dtype, tol):
    """Products whose bits differ, X among other factors, gates that end the holding, and reads between."""
    n = 17
    rng = numpy.random.default_rng(5)
    u = lambda: unitary(rng)    # noqa: E731
    mixed = lambda: [HM, XM, unitary(rng)][int(rng.integers(0, 3))]    # noqa: E731
    z = {(0, 8, 16): controlled(numpy.diag([1.0, -1.0]), 2)}
    seq = [layer(range(4, 17), n, u), z, layer(range(17), n, mixed), z, layer(range(17), n, mixed),
           {3: unitary(rng)}, layer(range(17), n, mixed), {(2, 5): CMat(XM)}, layer(range(2), n, u),
           layer(range(2, 9), n, u), z, layer(range(9), n, mixed), layer(range(12), n, mixed), z]
    for stop in range(1, len(seq) + 1):
        check(GpuBackend.make_state, n, seq[:stop], rng, dtype, tol)


@pytest.mark.parametrize("between", [False, True])
@pytest.mark.parametrize("entries,scale", [((1e200, 1e-200), 1e-300), ((1e-200, 1e200), 1e300), ((3e-160, 2.0), 1e200), ((1e300, 0.5), 1e-308),
                                           ((numpy.inf, 1.0), 1.0)])
def test_factors_near_the_limits_are_not_multiplied_together(entries, scale, between):
    """What two such products leave does not depend on whether the first was held: applied in turn they keep
    these amplitudes in range, their product would overflow or lose its bits."""
    n = 12
    rng = numpy.random.default_rng(3)
    v = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
    # the first qubit's halves at the scales that two applications bring back
    v.reshape(2, -1)[0] *= scale
    v.reshape(2, -1)[1] *= 1.0 / scale if entries[1] in (1e200, 1e-200) else 1.0
    step = {0: numpy.diag(entries), 7: HM}
    turn = {(0, 3): CMat(numpy.diag([1.0, 1j]))}
    out = []
    for flush in (True, False):
        be = GpuBackend.make_state(n, [], [])
        be.overwrite_relative_range(0, 2 ** n, v)
        for d in [step] + ([turn] if between else []) + [step]:
            be.kronselect_dot(d)
            if flush:
                be.flush()
        out.append(be.get_state())
        be.close()
    a, b = (x.view(numpy.float64) for x in out)
    assert numpy.array_equal(numpy.isnan(a), numpy.isnan(b)) and numpy.array_equal(numpy.isinf(a), numpy.isinf(b))
    if numpy.isfinite(entries[0]):
        assert numpy.isfinite(a).all() and a.any()
    # a rounding per factor and pass, against the largest amplitude of the half (H mixes amplitudes within one)
    for x, y in zip(a.reshape(2, -1), b.reshape(2, -1)):
        if numpy.isfinite(x).all():
            assert numpy.abs(x - y).max() <= 1e-14 * numpy.abs(x).max()

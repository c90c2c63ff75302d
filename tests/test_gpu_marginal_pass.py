"""The one-pass marginals (marked gpu): measured bits in a thread's registers (state bits 8..11), across lanes
(0..5), across waves (6, 7) and above a chunk, in any order, against numpy sums in complex128."""
import numpy
import pytest

from qip_amd import GpuBackend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n,bits", [
    (12, [0]), (12, [11]), (12, [6]), (12, [7]), (12, [6, 7]), (12, [7, 3, 9]), (12, list(range(12))),
    (12, [5, 8, 0, 10]), (12, [b for b in range(12) if b not in (6, 7)]), (12, [b for b in range(12) if b != 7]),
    (12, [b for b in range(12) if b not in (6, 8, 11)]), (13, [12]), (13, [12, 0, 6]), (13, list(range(13))),
    (16, [15, 1, 9, 6, 13]), (16, list(range(2, 16))[::-1]), (18, list(range(0, 18, 2))), (20, list(range(20))),
    (20, list(range(8, 20))), (20, list(range(12))), (21, [20, 19, 7, 6, 5, 4, 3, 2, 1, 0, 12, 11]),
])
def test_marginals_of_any_bits(n, bits, dtype):
    rng = numpy.random.default_rng(n * 100 + len(bits))
    psi = (rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)).astype(dtype)
    psi /= numpy.linalg.norm(psi)
    be = GpuBackend.make_state(n, [list(range(n))], [psi], statetype=dtype)
    held = psi.astype(dtype).astype(numpy.complex128)
    p = (held.real ** 2 + held.imag ** 2).reshape((2,) * n)
    qs = [n - 1 - b for b in bits]
    rest = tuple(q for q in range(n) if q not in qs)
    left = p.sum(axis=rest)                        # axes: the measured qubits, ascending
    order = [sorted(qs).index(q) for q in qs]      # axis of qs[j]
    want = left.transpose(order[::-1]).reshape(-1)   # qubit qs[j] on bit j
    got = be.measure_probabilities(qs)
    # each value is a sum of at most 2^21 non-negative terms, a few hundred roundings deep
    assert numpy.max(numpy.abs(got - want)) <= 2 ** -44 * numpy.max(want)
    assert numpy.array_equal(be.measure_probabilities(qs), got)
    be.close()

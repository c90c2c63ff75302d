"""The most likely outcome (marked gpu) by a maximum over chunks of 2^14: the first of equal values wins, wherever in a
lane, a wave, a workgroup or a later chunk it lies."""
import numpy
import pytest

from qip_amd import GpuBackend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 8, 9, 14, 15, 20, 22])
def test_first_of_the_largest(n):
    rng = numpy.random.default_rng(n)
    for places in (1, 2, 5):
        at = sorted(int(v) for v in rng.choice(2 ** n, size=min(places, 2 ** n), replace=False))
        psi = numpy.full(2 ** n, 0.25 / 2 ** (n / 2))
        psi[at] = 0.5
        be = GpuBackend.make_state(n, [list(range(n))], [psi])
        # the entwine order of all qubits: an outcome is the amplitude's index
        ms, ps = be.measure_probabilities(list(range(n)), top_k=1)
        assert ms == [at[0]] and ps == [0.25]
        rest = [q for q in range(n) if q != n // 2]
        if rest:
            marg = be.marginals(rest)
            ms, ps = be.measure_probabilities(rest, top_k=1)
            assert ms == [int(numpy.argmax(marg))] and ps == [float(marg.max())]
        be.close()

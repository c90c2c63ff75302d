"""Dense operators on 4 to 6 targets (marked gpu) at the edges of a wave's tile: fewer bases than one
tile holds, exactly one, the largest number of tiles that workgroups share and more than that (20 qubits); targets low, high
and scattered in an order of their own, with and without controls; against the oracle. Bars as for the
rest of the operator domain: 1e-12 (complex128), 2e-6 of the largest amplitude (complex64)."""
import numpy
import pytest

from oracle import oracle
from qip_amd import GpuBackend

pytestmark = pytest.mark.gpu


def unitary(rng, d):
    q, r = numpy.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
    return q * (numpy.diagonal(r) / numpy.abs(numpy.diagonal(r)))


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("k", [4, 5, 6])
@pytest.mark.parametrize("extra", [0, 1, 3, 4, 6, 8, 11, 15])
def test_tiles_of_every_size_against_the_oracle(k, extra, dtype):
    n = k + extra
    rng = numpy.random.default_rng(100 * k + extra)
    for where in ("low", "high", "scattered"):
        for controls in range(0, min(extra, 2) + 1):
            free = list(range(n))
            qs = {"low": free[n - k:], "high": free[:k], "scattered": sorted(rng.permutation(n)[:k].tolist())}[where]
            t = [int(q) for q in rng.permutation(qs)]              # the operator's own order of its targets
            c = [int(q) for q in rng.permutation([q for q in free if q not in t])[:controls]]
            print("dense tiles n", n, "targets", t, "controls", c, numpy.dtype(dtype).name, flush=True)
            psi = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
            psi /= numpy.linalg.norm(psi)
            u = unitary(rng, 2 ** k)
            be = GpuBackend.make_state(n, [free], [psi], statetype=dtype)
            be.apply_matrix(t, u, c)
            got = be.get_state().astype(numpy.complex128)
            be.close()
            full = u
            for _ in c:
                d = full.shape[0]
                full = numpy.block([[numpy.eye(d), numpy.zeros((d, d))], [numpy.zeros((d, d)), full]])
            want = numpy.zeros_like(psi)
            oracle.kronselect_dot({tuple(c + t): full}, psi, n, want, fast=True, nthreads=8)
            bar = 1e-12 if dtype == numpy.complex128 else 2e-6 * float(numpy.max(numpy.abs(want)))
            assert numpy.max(numpy.abs(got - want)) < bar

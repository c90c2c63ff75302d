"""Dense operators on 7 and 8 targets (marked gpu) as tiles in LDS and as the out-of-place product: fewer
tiles than the first needs, as many, and more than workgroups; targets low, high and scattered in an order of
their own, with and without controls; against numpy in complex128. Bars as for the operators on 4 to 6
targets: 1e-12 (complex128), 2e-6 of the largest amplitude (complex64)."""
import numpy
import pytest

from qip_amd import GpuBackend

pytestmark = pytest.mark.gpu


def unitary(rng, d):
    q, r = numpy.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
    return q * (numpy.diagonal(r) / numpy.abs(numpy.diagonal(r)))


def apply(psi, n, t, c, u):
    v = psi.reshape((2,) * n).copy()
    on = [slice(None)] * n
    for q in c:
        on[q] = 1
    k = len(t)
    axes = [q - sum(x < q for x in c) for q in t]
    out = numpy.tensordot(u.reshape((2,) * (2 * k)), v[tuple(on)], axes=(list(range(k, 2 * k)), axes))
    v[tuple(on)] = numpy.moveaxis(out, list(range(k)), axes)
    return v.reshape(-1)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("k", [7, 8])
@pytest.mark.parametrize("extra", [0, 2, 6, 12, 13, 14, 15])
def test_wide_tiles_of_every_size(k, extra, dtype):
    n = k + extra
    rng = numpy.random.default_rng(100 * k + extra)
    for where in ("low", "high", "scattered"):
        for controls in range(0, min(extra, 2) + 1):
            free = list(range(n))
            qs = {"low": free[n - k:], "high": free[:k], "scattered": sorted(rng.permutation(n)[:k].tolist())}[where]
            t = [int(q) for q in rng.permutation(qs)]              # the operator's own order of its targets
            c = [int(q) for q in rng.permutation([q for q in free if q not in t])[:controls]]
            print("wide tiles n", n, "targets", t, "controls", c, numpy.dtype(dtype).name, flush=True)
            psi = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
            psi /= numpy.linalg.norm(psi)
            u = unitary(rng, 2 ** k)
            be = GpuBackend.make_state(n, [free], [psi], statetype=dtype)
            be.apply_matrix(t, u, c)
            got = be.get_state().astype(numpy.complex128)
            be.close()
            want = apply(psi, n, t, c, u)
            bar = 1e-12 if dtype == numpy.complex128 else 2e-6 * float(numpy.max(numpy.abs(want)))
            assert numpy.max(numpy.abs(got - want)) < bar

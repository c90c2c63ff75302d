"""Dense operators on the four lowest state bits (marked gpu): on states of more than 512 tiles a kernel of their own,
below that the kernel that every other place of four targets takes. Against numpy in complex128."""
import numpy
import pytest

from qip_amd import CMat, GpuBackend

pytestmark = pytest.mark.gpu


def expected(psi, n, targets, controls, u):
    v = psi.reshape((2,) * n)
    on = [slice(None)] * n
    for q in controls:
        on[q] = 1
    sub = v[tuple(on)]
    axes = [q - sum(c < q for c in controls) for q in targets]
    k = len(targets)
    out = numpy.tensordot(u.reshape((2,) * (2 * k)), sub, axes=(list(range(k, 2 * k)), axes))
    v = v.copy()
    v[tuple(on)] = numpy.moveaxis(out, list(range(k)), axes)
    return v.reshape(-1)


@pytest.mark.parametrize("dtype", [numpy.complex128, numpy.complex64])
@pytest.mark.parametrize("n,order,control_bits", [
    (19, [3, 2, 1, 0], []),               # 512 tiles
    (20, [3, 2, 1, 0], []),               # 1024: one step of every wave
    (20, [0, 2, 3, 1], []),
    (20, [1, 3, 0, 2], [4]),              # 512 again
    (21, [2, 0, 1, 3], [4]),
    (21, [3, 0, 2, 1], [20]),
    (22, [0, 1, 2, 3], [5, 9]),
    (22, [3, 1, 2, 0], [4, 21]),
    (23, [2, 3, 0, 1], []),               # several tiles a wave, odd ends
    (21, [4, 3, 2, 1], []),               # one bit higher: the other kernel
])
def test_four_lowest_bits(n, order, control_bits, dtype):
    rng = numpy.random.default_rng(n + sum(order[:2]))
    print("four low targets", n, order, control_bits, numpy.dtype(dtype).name, flush=True)
    psi = (rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)).astype(dtype)
    u = rng.standard_normal((16, 16)) + 1j * rng.standard_normal((16, 16))      # row and column order matter
    targets, controls = [n - 1 - b for b in order], [n - 1 - b for b in control_bits]
    be = GpuBackend.make_state(n, [], [], statetype=dtype)
    be.overwrite_relative_range(0, 2 ** n, psi)
    m = u
    for _ in controls:
        m = CMat(m)
    want = psi.astype(numpy.complex128)
    for _ in range(2):
        be.kronselect_dot({tuple(controls + targets): m})
        want = expected(want, n, targets, controls, u)
        if dtype == numpy.complex64:
            want = want.astype(dtype).astype(numpy.complex128)
    # a group of 16 amplitudes: |U| times their norm bounds every partial sum; three real products of 16 terms each, and
    # the second application carries the first one's error through U again
    eps = numpy.finfo(numpy.float64).eps
    norm = numpy.linalg.norm(u, 2)
    bound = 2 * 4 * 16 * eps * norm ** 2 * 16 * numpy.abs(psi).max()
    if dtype == numpy.complex64:
        # its state rounds what may differ in the last bit of FP64: one unit of single precision, twice
        bound += 4 * numpy.finfo(numpy.float32).eps * norm * numpy.abs(want).max()
    assert numpy.abs(be.get_state() - want).max() <= bound
    be.close()

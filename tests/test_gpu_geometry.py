"""The tile shape of complex64 flushes: 8 amplitudes per thread while a flush
has at most 512 tiles, 16 above; on both sides of the line against the
same shape asked for, and against the complex128 state."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, gate_matrix
from q1tsim_amd import workloads

pytestmark = pytest.mark.gpu


def run(ops, amps, prec, geometry=None):
    g = GpuVectorState.from_amplitudes(amps, 1, prec)
    if geometry:
        g.set_geometry(*geometry)
    for name, q, p in ops:
        g.apply_gate(gate_matrix(name, p), q)
    g.flush()
    return g.column(0)


@pytest.mark.parametrize("n,shape", [(14, (12, 3, 4)), (15, (12, 3, 4)), (21, (12, 3, 4)), (22, (12, 4, 4))])
def test_shape_by_number_of_tiles(n, shape):
    ops = workloads.random_layered(n, 6, n)
    rng = np.random.Generator(np.random.PCG64(n))
    amps = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)).astype(np.complex64)
    amps = amps / np.linalg.norm(amps)
    got = run(ops, amps, "c64")
    assert np.array_equal(got, run(ops, amps, "c64", shape))
    # at most 4 roundings of values of magnitude <= max per gate and 2 to read in
    ref = run(ops, amps, "c128")
    assert np.max(np.abs(got - ref)) <= (4 * len(ops) + 2) * 2.0**-24 * np.max(np.abs(ref))

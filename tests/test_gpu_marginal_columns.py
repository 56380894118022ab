"""Marginals of states with several columns, on both sides of the number of
shares from which they are added by a launch of their own: each column's weight
has the bits that the column gives in a state of its own, through the item
queue and through the allocation-free entry point."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, Xoshiro

pytestmark = pytest.mark.gpu


# (n, measured qubits): columns of one share, 128 to 1024 shares in all
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,nm", [(11, 7), (14, 5), (16, 3), (16, 5), (16, 6), (18, 3), (18, 4), (20, 1), (20, 2), (20, 3)])
def test_columns_as_on_their_own(n, nm, precision):
    shots = 32 << nm
    rng = np.random.Generator(np.random.PCG64([n, nm]))
    a = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    s = GpuVectorState.from_amplitudes(a / np.linalg.norm(a), shots, precision)
    res, x = np.zeros(shots, np.uint64), Xoshiro(n)
    for q in range(nm):
        s.measure_into(q, q, res, x)
    assert s.ncols == 1 << nm
    qubits = (0, nm, n - 1)
    got = [s.marginal_w0(q) for q in qubits]
    if s.ncols <= 256:
        for q, w in zip(qubits, got):
            assert np.array_equal(s.marginal_w0_noalloc(q), w)
    for c in range(0, s.ncols, max(1, s.ncols // 8)):
        one = GpuVectorState.from_amplitudes(s.column(c), 1, precision)
        for q, w in zip(qubits, got):
            assert one.marginal_w0(q)[0] == w[c]
        one.close()
    s.close()

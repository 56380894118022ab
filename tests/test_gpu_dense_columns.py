"""Dense gates on 4, 5 and 6 qubits of small states with many branch columns
against the dense simulator: the states have fewer free index bits than
k_dense_tile needs, and the columns make enough blocks for k_dense_rows to give
a wave several of the matrix's row tiles (1, 2 and 4 at these widths)."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, Xoshiro
from tests.golden import dense_sim

pytestmark = pytest.mark.gpu


def unitary(rng, d):
    a, b, c = np.exp(2j * np.pi * rng.uniform(size=(3, d)))
    return np.ascontiguousarray(a[:, None] * np.fft.ifft(b[:, None] * np.fft.fft(np.diag(c), axis=0), axis=0))


# (n, k, measured qubits): 2^measured columns; below, at and above the counts
# from which a wave would take two and four row tiles
SIZES = [(12, 4, 6), (12, 4, 7), (12, 4, 8), (11, 4, 7), (11, 4, 8), (11, 4, 9), (10, 4, 9), (12, 5, 7), (12, 5, 8),
         (11, 5, 9), (10, 5, 9), (10, 6, 8)]


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,k,nm", SIZES)
def test_dense_gate_on_many_columns(n, k, nm, precision):
    rng = np.random.Generator(np.random.PCG64([n, k, nm]))
    shots = 32 << nm
    # a random product state: measuring qubit q leaves the others' amplitudes
    a = np.ones(1)
    for _ in range(n):
        t, p = rng.uniform(0.24 * np.pi, 0.26 * np.pi), rng.uniform(0, 2 * np.pi)
        a = np.kron(a, [np.cos(t), np.exp(1j * p) * np.sin(t)])
    g = GpuVectorState.from_amplitudes(a, shots, precision)
    res, x = np.zeros(shots, np.uint64), Xoshiro(n + nm)
    for q in range(nm):
        g.measure_into(q, q, res, x)
    assert g.ncols == 1 << nm
    cols = g.states
    m, bits = unitary(rng, 1 << k), [int(b) for b in rng.permutation(n)[:k]]
    g.apply_gate(m, bits)
    ref = np.stack([dense_sim.apply(cols[:, c], m, bits, n) for c in range(cols.shape[1])], axis=1)
    # 2^(k+1) products per part, each sum of magnitude <= 1 accumulated in the
    # state's precision
    tol = 2.0 ** (k + 1) * (2.0 ** -53 if precision == "c128" else 2.0 ** -24)
    assert np.abs(g.states - ref).max() <= tol
    g.close()

"""Dense gates on 4..12 qubits (dense.hip) against the dense simulator: both
kernels (whole-row tiles; up to 8 columns with the rows split over several
workgroups), sizes around the switch between them, the smallest state each
width allows, targets in the lowest, highest and scattered bits, controls
found from the matrix inside and outside the tile, several columns."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, Xoshiro
from tests.golden import dense_sim

pytestmark = pytest.mark.gpu


def unitary(rng, d):
    a, b, c = np.exp(2j * np.pi * rng.uniform(size=(3, d)))
    return np.ascontiguousarray(a[:, None] * np.fft.ifft(b[:, None] * np.fft.fft(np.diag(c), axis=0), axis=0))


def tol(precision, k):
    # 2^(k+1) products per part, each sum of magnitude <= 1 accumulated in the
    # state's precision: absolute error below 2^(k+1) * 2^-53 (2^-24)
    return 2.0 ** (k + 1) * (2.0 ** -53 if precision == "c128" else 2.0 ** -24)


def amplitudes(rng, n):
    a = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return a / np.linalg.norm(a)


# (n, k, controls): k alone, k + few, across the tile / row-split switch
SIZES = [(4, 4, 0), (5, 4, 1), (12, 4, 0), (13, 4, 0), (15, 4, 2), (6, 5, 1), (13, 5, 0), (16, 5, 3), (6, 6, 0),
         (13, 6, 0), (17, 6, 0), (18, 6, 2), (7, 7, 0), (12, 7, 0), (18, 7, 1), (8, 8, 0), (12, 8, 1), (17, 8, 0),
         (18, 8, 0), (9, 9, 0), (13, 9, 2), (18, 9, 0), (10, 10, 0), (14, 10, 2), (18, 10, 0), (11, 11, 0),
         (13, 11, 1), (12, 12, 0), (14, 12, 0)]


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,k,nc", SIZES)
def test_dense_gate(n, k, nc, precision):
    rng = np.random.Generator(np.random.PCG64([n, k, nc]))
    a = amplitudes(rng, n)
    places = [[int(b) for b in rng.permutation(n)[:k + nc]]]
    places.append(list(range(n - k - nc, n)))   # the lowest index bits
    places.append(list(range(k + nc))[::-1])    # the highest
    g = GpuVectorState.from_amplitudes(a, 1, precision)
    ref = a if precision == "c128" else a.astype(np.complex64).astype(np.complex128)
    for bits in places:
        u = unitary(rng, 1 << k)
        m = np.eye(1 << (k + nc), dtype=complex)
        m[-(1 << k):, -(1 << k):] = u
        g.apply_gate(m, bits)
        ref = dense_sim.apply(ref, m, bits, n)
    assert np.abs(g.column(0) - ref).max() <= 3 * tol(precision, k)
    g.close()


def test_dense_gate_on_columns():
    n, shots = 9, 200
    rng = np.random.Generator(np.random.PCG64(1))
    g = GpuVectorState.from_amplitudes(amplitudes(rng, n), shots)
    res, x = np.zeros(shots, np.uint64), Xoshiro(2)
    for q in (0, 4, 8):
        g.measure_into(q, q, res, x)
    cols = g.states
    assert cols.shape[1] > 4
    for k in (3, 4, 6, 8):
        u, bits = unitary(rng, 1 << k), [int(b) for b in rng.permutation(n)[:k]]
        g.apply_gate(u, bits)
        cols = np.stack([dense_sim.apply(cols[:, c], u, bits, n) for c in range(cols.shape[1])], axis=1)
    assert np.abs(g.states - cols).max() <= 4 * tol("c128", 8)
    g.close()

"""Short runs of gates on states below 14 qubits go to single-gate kernels, longer
ones to a whole-state program: the amplitudes are the same bits whichever way
the runs are cut, for every gate form, width and precision, alone and between
dense two-qubit gates, and with several columns."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, Xoshiro, gate_matrix

pytestmark = pytest.mark.gpu

NAMES = [("h", 1, 0), ("x", 1, 0), ("y", 1, 0), ("z", 1, 0), ("s", 1, 0), ("t", 1, 0), ("v", 1, 0), ("rx", 1, 1),
         ("ry", 1, 1), ("rz", 1, 1), ("u1", 1, 1), ("u2", 1, 2), ("u3", 1, 3), ("cx", 2, 0), ("cy", 2, 0), ("cz", 2, 0),
         ("ch", 2, 0), ("crx", 2, 1), ("crz", 2, 1), ("cu1", 2, 1), ("cu3", 2, 3), ("swap", 2, 0), ("ccx", 3, 0)]


def gates(n, count, seed):
    rng = np.random.Generator(np.random.PCG64([n, seed]))
    out = []
    while len(out) < count:
        name, k, npar = NAMES[len(out) % len(NAMES) if n > 2 else int(rng.integers(13))]
        if k <= n:
            out.append((gate_matrix(name, list(rng.uniform(0, 6.3, npar))), [int(b) for b in rng.permutation(n)[:k]]))
    return out


def prepared(n, precision, columns):
    rng = np.random.Generator(np.random.PCG64([n, columns]))
    a = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    s = GpuVectorState.from_amplitudes(a / np.linalg.norm(a), 64, precision)
    res, x = np.zeros(64, np.uint64), Xoshiro(5)
    for q in range(columns):
        s.measure_into(q, q, res, x)
    return s


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,columns", [(1, 0), (2, 0), (5, 0), (8, 3), (11, 0), (12, 0), (12, 2), (13, 0)])
def test_runs_cut_anywhere(n, columns, precision):
    gs = gates(n, 46, 1)
    states = [prepared(n, precision, columns) for _ in range(7)]
    for run, s in zip((46, 1, 2, 3, 4, 5, 7), states):
        for k in range(0, len(gs), run):
            for m, bits in gs[k:k + run]:
                s.apply_gate(m, bits)
            s.flush()
    want = states[0].states
    for s in states[1:]:
        assert np.array_equal(s.states, want)
        s.close()


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [2, 8, 12, 13])
def test_runs_between_dense_pairs(n, precision):
    # a state with flush graphs keeps every run in a whole-state program
    a, b = prepared(n, precision, 0), prepared(n, precision, 0)
    b.set_graph(True)
    rng = np.random.Generator(np.random.PCG64(n))
    for k in range(1, 7):
        u, _ = np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))
        run = gates(n, k, k)
        for s in (a, b):
            s.apply_gate(np.ascontiguousarray(u), [0, n - 1])
            for m, bits in run:
                s.apply_gate(m, bits)
    for s in (a, b):
        s.flush()
    assert 0 < a.stats()["phases"] < b.stats()["phases"]
    assert np.array_equal(a.column(0), b.column(0))
    a.close()
    b.close()


@pytest.mark.parametrize("precision,n,lone", [("c128", 5, 2), ("c128", 11, 2), ("c128", 12, 3), ("c128", 13, 4),
                                              ("c64", 11, 2), ("c64", 12, 2), ("c64", 13, 3)])
def test_route_of_a_flush(precision, n, lone):
    s = prepared(n, precision, 0)
    for count in (1, lone, lone + 1):
        for m, bits in gates(n, count, 2):
            s.apply_gate(m, bits)
        s.flush()
        # register phases: of whole-state programs only
        assert (s.stats()["phases"] > 0) == (count > lone)
    s.close()

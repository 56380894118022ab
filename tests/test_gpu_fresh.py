"""Flushes of a state that is still |0..0>: the sweeps start without its
amplitudes in memory and skip the tiles that no gate has reached.  The result
is that of the same gates on |0..0> given as amplitudes: whole states in LDS
(1 to 13 qubits), tiles, gates that reach every bit and few of them, controls
and phases on untouched bits, gates that no sweep takes first, between and
last, specialised kernels with and without prefetch, a captured flush, and a
second flush and a reset after the first."""
import numpy as np
import pytest

from q1tsim_amd import workloads
from q1tsim_amd.gvs import GpuVectorState, gate_matrix

pytestmark = pytest.mark.gpu


def dense4(seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return np.linalg.qr(rng.normal(size=(16, 16)) + 1j * rng.normal(size=(16, 16)))[0]


def circuit(kind, n):
    if kind == "layers":
        return [(gate_matrix(g, p), q) for g, q, p in workloads.random_layered(n, 8, n)]
    if kind == "few":        # three qubits at the ends, controls and phases on bits that stay 0
        g = [(gate_matrix("h"), [q]) for q in {0, n // 2, n - 1}]
        if n > 1:
            g += [(gate_matrix("cx"), [0, n - 1])] + \
                [(gate_matrix("crz", [0.3 + q]), [q, (q + 1) % n]) for q in range(n)]
        return g
    if kind == "x":          # basis states: each bit set in turn, far bits first
        return [(gate_matrix("x"), [q]) for q in range(n)] + [(gate_matrix("t"), [0])]
    bits = [[0, 1, n - 2, n - 1], [n // 2, 0, 1, n - 1], list(range(4))]
    place = {"dense_first": (0,), "dense_between": (n // 2,), "dense_last": (10 ** 9,), "dense_all": (0, n, 10 ** 9)}[kind]
    g = [(gate_matrix("h"), [q]) for q in range(n)] + [(gate_matrix("cx"), [q, q + 1]) for q in range(n - 1)]
    for k, at in enumerate(place):
        g.insert(min(at, len(g)), (dense4(k), bits[k % 3]))
    return g


def run(s, gates):
    for m, q in gates:
        s.apply_gate(m, q)
    s.flush()
    return s.column(0)


KINDS = ["layers", "few", "x", "dense_first", "dense_between", "dense_last", "dense_all"]


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,kind", [(n, k) for n in (1, 3, 5, 11, 13, 14, 17, 22) for k in KINDS
                                    if n > 3 or k in ("few", "x")])
def test_fresh_equals_dense(n, kind, precision):
    gates = circuit(kind, n)
    zero = np.zeros(1 << n, complex)
    zero[0] = 1
    want = run(GpuVectorState.from_amplitudes(zero, 1, precision), gates)
    s = GpuVectorState(n, 1, precision)
    assert np.array_equal(run(s, gates), want)
    s.reset_all()
    assert np.array_equal(s.column(0), zero)
    assert np.array_equal(run(s, gates), want)
    # a second flush goes on from the first
    more = circuit("few", n)
    d = GpuVectorState.from_amplitudes(zero, 1, precision)
    run(d, gates)
    assert np.array_equal(run(s, more), run(d, more))


@pytest.mark.parametrize("precision,geometry", [("c128", (12, 4, 4)), ("c64", (12, 3, 4)), ("c64", (13, 4, 5))])
@pytest.mark.parametrize("kind", ["layers", "few", "dense_between"])
def test_fresh_by_every_route(kind, precision, geometry):
    n = 16
    gates = circuit(kind, n)
    zero = np.zeros(1 << n, complex)
    zero[0] = 1
    for setup in (lambda s: None, lambda s: s.set_jit(True), lambda s: s.set_jit(True, factors=False),
                  lambda s: s.set_jit(True, prefetch=True), lambda s: s.set_graph(True), lambda s: s.set_plan(4, True),
                  lambda s: s.set_plan(0, False)):
        out = []
        for s in (GpuVectorState.from_amplitudes(zero, 1, precision), GpuVectorState(n, 1, precision)):
            s.set_geometry(*geometry)
            setup(s)
            out.append(run(s, gates))
            s.close()
        assert np.array_equal(out[0], out[1])

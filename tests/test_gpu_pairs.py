"""Dense two-qubit gates inside sweeps: against the same gates one launch each.
Pairs on every kind of bits (both low, both high, adjacent, either order),
between one-qubit gates and controlled gates on their bits, alone in a flush,
from |0..0>, on several columns and tile shapes, interpreted and specialised,
and with matrices that are not unitary."""
import numpy as np
import pytest

from q1tsim_amd import workloads
from q1tsim_amd.gvs import GpuVectorState, gate_matrix

pytestmark = pytest.mark.gpu


def pair(rng):
    return np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))[0]


def gates(n, count, kind):
    rng = np.random.Generator(np.random.PCG64([n, count]))
    out = []
    if kind == "one":
        return [(pair(rng), [n - 1, 0])]
    for k in range(count):
        q = [int(b) for b in rng.permutation(n)[:2]]
        if k % 7 == 0:
            q = [[0, 1], [1, 0], [n - 1, n - 2], [0, n - 1], [n // 2, n // 2 - 1]][k // 7 % 5]
        out.append((pair(rng), q))
        if kind == "mixed":
            for name in ("h", "rz", "cx", "cu1", "x", "swap", "rx"):
                p = [float(rng.uniform(0, 6))] if name in ("rz", "cu1", "rx") else []
                w = 2 if name in ("cx", "cu1", "swap") else 1
                if rng.uniform() < 0.4:
                    out.append((gate_matrix(name, p), [int(b) for b in rng.permutation(n)[:w]]))
    return out


def run(n, ops, prec, setup, fresh=False, cols=1):
    rng = np.random.Generator(np.random.PCG64(n))
    a = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)).astype(np.complex64).astype(complex)
    s = GpuVectorState(n, 2, prec) if fresh else GpuVectorState.from_amplitudes(a / np.linalg.norm(a), 2, prec)
    if cols == 2:
        s.apply_conditional_gate([0, 1], gate_matrix("h"), [n // 2])
    setup(s)
    for m, q in ops:
        s.apply_gate(m, q)
    s.flush()
    out = s.states.copy(), s.stats()
    s.close()
    return out


# a pair rounds each of its values at most 8 times on each side, others fewer;
# values stay below the norm, which is 1
def tol(prec, ops):
    return 16 * len(ops) * (2.0 ** -53 if prec == "c128" else 2.0 ** -24)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,count,kind,fresh,cols", [(14, 1, "one", False, 1), (14, 60, "pairs", True, 1),
                                                     (15, 50, "mixed", False, 2), (18, 90, "pairs", False, 1),
                                                     (18, 40, "mixed", True, 1), (22, 30, "mixed", False, 1)])
def test_pairs_in_sweeps(n, count, kind, fresh, cols, prec):
    ops = gates(n, count, kind)
    ref, _ = run(n, ops, prec, lambda s: s.set_plan(0, False), fresh, cols)
    got, st = run(n, ops, prec, lambda s: None, fresh, cols)
    assert np.abs(got - ref).max() <= tol(prec, ops)
    assert st["launches"] == 1 if kind == "one" else st["launches"] < len(ops) // 2


@pytest.mark.parametrize("prec,geometry", [("c128", (12, 3, 4)), ("c128", (12, 4, 4)), ("c64", (12, 3, 4)),
                                           ("c64", (12, 4, 4)), ("c64", (13, 4, 5))])
def test_pairs_by_every_kernel(prec, geometry):
    n = 16
    ops = gates(n, 40, "mixed")
    ref, _ = run(n, ops, prec, lambda s: s.set_plan(0, False))
    for jit in (None, {}, {"factors": False}, {"prefetch": True}):
        def setup(s):
            if jit is not None:
                s.set_jit(True, **jit)
            s.set_geometry(*geometry)
        for fresh in (False, True):
            want = run(n, ops, prec, lambda s: s.set_plan(0, False), True)[0] if fresh else ref
            assert np.abs(run(n, ops, prec, setup, fresh)[0] - want).max() <= tol(prec, ops)


def test_pairs_beside_graphs_and_fusion():
    n = 16
    ops = gates(n, 25, "mixed")
    for prec, setup in (("c128", lambda s: s.set_graph(True)), ("c64", lambda s: s.set_plan(4, True)),
                        ("c64", lambda s: s.set_graph(True))):
        ref, _ = run(n, ops, prec, lambda s: s.set_plan(0, False))
        assert np.abs(run(n, ops, prec, setup)[0] - ref).max() <= tol(prec, ops)


def test_a_pair_that_is_not_unitary():
    n = 14
    ops = gates(n, 6, "mixed")
    ops.insert(4, (np.arange(16).reshape(4, 4) * (0.01 + 0.02j), [3, 11]))   # norm below 1
    ref, _ = run(n, ops, "c128", lambda s: s.set_plan(0, False))
    assert np.abs(run(n, ops, "c128", lambda s: None)[0] - ref).max() <= tol("c128", ops)

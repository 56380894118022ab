"""Reduced sweep programs (reduce_program): gates without their larger entry,
diagonal gates as phases and factors gathered per thread, the common factor
applied once.  Against the same gates one launch each: every form at angles
where either entry is the larger one, zero or equal, more gates than a factor
is carried over (80 complex64, 800 complex128), controls on register, thread
and outer bits between them, matrices that are not unitary (inside and outside
of what is reduced), several columns, and every kernel that runs programs."""
import math

import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, gate_matrix

pytestmark = pytest.mark.gpu

ANGLES = [0.0, math.pi / 2, math.pi, 3 * math.pi / 2, 2 * math.pi, 1e-9, math.pi - 1e-9, -0.4]
ONE = ["h", "rx", "ry", "rz", "s", "t", "u1", "x", "y", "z", "u3", "sdg", "v"]
TWO = ["cx", "cz", "crx", "cry", "crz", "ch", "cu1", "swap"]
PARAMS = {"rx": 1, "ry": 1, "rz": 1, "u1": 1, "u3": 3, "crx": 1, "cry": 1, "crz": 1, "cu1": 1}


def gates(n, count, seed, kind):
    rng = np.random.Generator(np.random.PCG64([n, seed]))
    out = []
    while len(out) < count:
        names = {"mixed": ONE + ONE + TWO, "dense": ["h", "rx", "ry"], "diag": ["rz", "t", "cu1", "crz", "h"]}[kind]
        name = names[int(rng.integers(len(names)))]
        par = [float(rng.uniform(0, 6.3)) if rng.uniform() < 0.6 else ANGLES[int(rng.integers(len(ANGLES)))]
               for _ in range(PARAMS.get(name, 0))]
        k = 2 if name in TWO else 1
        out.append((gate_matrix(name, par), [int(b) for b in rng.permutation(n)[:k]]))
    return out


def run(n, amps, ops, prec, setup, cols=1):
    s = GpuVectorState.from_amplitudes(amps, 2, prec)
    if cols == 2:
        s.apply_conditional_gate([0, 1], gate_matrix("h"), [n // 2])
    setup(s)
    for m, q in ops:
        s.apply_gate(m, q)
    s.flush()
    out = s.states.copy()
    s.close()
    return out


def start(n):
    rng = np.random.Generator(np.random.PCG64(n))
    a = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)).astype(np.complex64).astype(complex)
    return a / np.linalg.norm(a)


# a gate rounds each of its values at most 4 times, on each side, and they
# stay below the norm, which is 1
def tol(prec, count):
    return 8 * count * (2.0 ** -53 if prec == "c128" else 2.0 ** -24)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,count,kind", [(14, 1700, "dense"), (14, 300, "mixed"), (15, 400, "diag"), (17, 300, "mixed"),
                                          (22, 120, "mixed")])
def test_reduced_programs(n, count, kind, prec):
    ops = gates(n, count, 1, kind)
    ref = run(n, start(n), ops, prec, lambda s: s.set_plan(0, False))
    got = run(n, start(n), ops, prec, lambda s: None)
    assert np.abs(got - ref).max() <= tol(prec, count)


@pytest.mark.parametrize("prec,geometry", [("c128", (12, 3, 4)), ("c128", (12, 4, 4)), ("c64", (12, 3, 4)),
                                           ("c64", (12, 4, 4)), ("c64", (13, 4, 5))])
def test_every_kernel(geometry, prec):
    n, count = 16, 250
    ops = gates(n, count, 2, "mixed")
    ref = run(n, start(n), ops, prec, lambda s: s.set_plan(0, False), cols=2)
    assert ref.shape[1] == 2
    for jit in ({}, {"on": True}, {"on": True, "factors": False}, {"on": True, "prefetch": True}):
        def setup(s):
            if jit:
                s.set_jit(**jit)
            s.set_geometry(*geometry)
        assert np.abs(run(n, start(n), ops, prec, setup, cols=2) - ref).max() <= tol(prec, count)


@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_matrices_that_are_not_unitary(prec):
    n = 14
    ops = gates(n, 40, 3, "mixed")
    for k, f in enumerate((0.9, 1.1, 0.5, 3.0, 0.9j)):   # a growth of 1.34 in all
        for j, name in enumerate(("h", "rx", "ry", "rz")):
            ops.insert(7 * k + j, (f * gate_matrix(name, [0.3 + k] if j else []), [(3 * k + j) % n]))
    ops.insert(20, (np.zeros((2, 2)), [3]))
    ref = run(n, start(n), ops[:20], prec, lambda s: s.set_plan(0, False))
    got = run(n, start(n), ops[:20], prec, lambda s: None)
    assert np.abs(got - ref).max() <= 200 * tol(prec, 20)   # the norm stays below 3^4 * 1.1^8 < 200
    assert not run(n, start(n), ops, prec, lambda s: None).any()

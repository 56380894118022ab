"""Circuits wide enough for tile sweeps give the same states in a batch and
alone up to rounding: alone they run reduced programs on searched tiles, in a
batch the gates' own forms (complex64: on greedy tiles), so the gates' rounding
differs in place and order.  Smaller states run the same programs either way and
agree bit for bit."""
import numpy as np
import pytest

from q1tsim_amd import workloads
from q1tsim_amd.q1tsim import Batch, Circuit

pytestmark = pytest.mark.gpu

SHOTS = 64
WL = [(n, nc, prog[:-1], s) for (n, nc, prog, s) in   # stop before measure_all
      workloads.batch_workload(8, seed=23, qubits=(14, 18), depths=(8, 14), meas=(1, 3))]


def make(n, nc, prog, seed, prec):
    c = Circuit(n, nc)
    workloads.build_program(c, prog)
    c.set_backend(prec)
    c.seed(seed)
    return c


@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_states_in_a_batch_and_alone(prec):
    batch = Batch(prec)
    circs = [make(n, nc, prog, s, prec) for (n, nc, prog, s) in WL]
    for c in circs:
        batch.add(c)
    batch.execute(SHOTS, keep_states=True)
    eps = 2.0 ** -53 if prec == "c128" else 2.0 ** -24
    for (n, nc, prog, s), c in zip(WL, circs):
        solo = make(n, nc, prog, s, prec)
        solo.execute(SHOTS)
        # a draw that falls between the two runs' weights would differ: within
        # 1e-6 of an edge in complex64, absent for these seeds
        assert c.counts() == solo.counts(), (n, s)
        # an op (gate, collapse) moves a column by at most 6 eps of its norm in
        # either run: two products and a sum per part of each amplitude of a pair
        tol = 2 * 6 * eps * len(prog)
        for col in range(c.nr_columns()):
            d = np.linalg.norm(c.amplitudes(col) - solo.amplitudes(col))
            assert d <= tol, (n, s, col, d, tol)


@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_small_states_in_a_batch_and_alone(prec):
    wl = [(n, nc, prog[:-1], s) for (n, nc, prog, s) in
          workloads.batch_workload(12, seed=29, qubits=(3, 13), depths=(3, 12), meas=(1, 3))]
    batch = Batch(prec)
    circs = [make(n, nc, prog, s, prec) for (n, nc, prog, s) in wl]
    for c in circs:
        batch.add(c)
    batch.execute(SHOTS, keep_states=True)
    for (n, nc, prog, s), c in zip(wl, circs):
        solo = make(n, nc, prog, s, prec)
        solo.execute(SHOTS)
        assert c.counts() == solo.counts(), (n, s)
        for col in range(c.nr_columns()):
            assert np.array_equal(c.amplitudes(col), solo.amplitudes(col)), (n, s, col)

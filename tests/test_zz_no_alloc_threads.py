"""Allocation-free marginals called from several threads at once, each thread
with a state of its own (sizes of one workgroup per column and of many, both
precisions, one column and several): every call gives the bits of
q1t_gvs_marginal_w0, and so do the calls that come after."""
import threading

import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState, Xoshiro

pytestmark = pytest.mark.gpu


def prepared(n, precision, nm, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    a = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    s = GpuVectorState.from_amplitudes(a / np.linalg.norm(a), 256, precision)
    res, x = np.zeros(256, np.uint64), Xoshiro(seed)
    for q in range(nm):
        s.measure_into(q, q, res, x)
    return s


def test_noalloc_marginals_of_several_threads():
    states = [prepared(20, "c128", 0, 1), prepared(16, "c64", 3, 2), prepared(9, "c128", 5, 3),
              prepared(18, "c64", 1, 4)]
    expected = [[s.marginal_w0(q) for q in range(s.nr_bits)] for s in states]
    wrong, start = [], threading.Barrier(len(states))

    def work(i):
        start.wait()
        for k in range(200):
            q = k % states[i].nr_bits
            if not np.array_equal(states[i].marginal_w0_noalloc(q), expected[i][q]):
                wrong.append((i, k, q))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(states))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:10]
    for s, exp in zip(states, expected):
        for q in range(s.nr_bits):
            assert np.array_equal(s.marginal_w0_noalloc(q), exp[q])
        s.close()

"""The sampling tree and walk (items.hip) against the oracle, index by index:
widths at which a level is added (5, 9, 13, 17 qubits), one workgroup's 4096
inputs, a second launch of levels (13 qubits and up), one column and several,
and more uniforms and results than are read from and written to host memory
(2^17 runs)."""
import numpy as np
import pytest

from oracle import oracle as orc
from q1tsim_amd.gvs import GpuVectorState, gate_matrix

pytestmark = pytest.mark.gpu


def expect(s, n, u):
    out, off = [], 0
    for c, cnt in enumerate(s.counts):
        idx, _ = orc.tree_sample_many(orc.canonical_weights(s.column(c)), u[off:off + cnt])
        out += [orc.reverse_bits(int(k), n) for k in np.sort(idx)]
        off += cnt
    return np.array(out, np.uint64)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,runs,split", [(1, 300, 0), (3, 256, 2), (4, 257, 0), (5, 300, 3), (8, 300, 0), (9, 300, 2),
                                          (12, 300, 3), (13, 300, 0), (13, 300, 2), (16, 1000, 0), (17, 1000, 3),
                                          (21, 300, 0), (6, 1 << 17, 2), (14, (1 << 17) + 1, 0)])
def test_samples(n, runs, split, precision):
    rng = np.random.Generator(np.random.PCG64([n, runs]))
    s = GpuVectorState(n, runs, precision)
    s.set_random_normal(n)
    for k in range(split):   # columns: a gate on every second, third, ... run
        ctrl = (np.arange(runs) // max(1, runs // (3 * (k + 1))) % 2).astype(np.uint8)
        s.apply_conditional_gate(ctrl, gate_matrix("h"), [k % n])
    s.flush()
    assert (len(s.counts) > 1) == (split > 0)
    for _ in range(2):
        u = rng.uniform(size=runs)
        res = np.zeros(runs, np.uint64)
        s.measure_all_uniforms(list(range(n)), u, res, collapse=False)
        assert np.array_equal(res, expect(s, n, u))
    s.close()

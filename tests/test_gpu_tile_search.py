"""When the default plan searches tiles: always with register programs and
blocks of up to 4 qubits, with blocks of 5 and 6 qubits from 128 MiB (24 qubits
complex64) on.  A searched plan needs fewer sweeps than the greedy one, so the
sweeps of a flush tell which it was; the states agree to FP32 rounding."""
import numpy as np
import pytest

from q1tsim_amd import workloads
from q1tsim_amd.gvs import GpuVectorState

pytestmark = pytest.mark.gpu


def run(n, fusion_k, mode):
    ops = workloads.random_layered(n, 12, n)
    s = GpuVectorState(n, 1, "c64")
    s.set_plan(fusion_k, True)
    if mode is not None:
        s.set_plan_search(mode)
    for name, bits, par in ops:
        s.apply_named(name, bits, par)
    s.flush()
    sweeps, a = s.stats()["sweeps"], s.column(0) if n <= 20 else None
    s.close()
    return sweeps, a, len(ops)


@pytest.mark.parametrize("n,fusion_k,searched", [(20, 0, True), (20, 4, True), (18, 5, False), (20, 5, False),
                                                 (20, 6, False), (23, 6, False), (24, 5, True), (24, 6, True)])
def test_default_tile_search(n, fusion_k, searched):
    got, a, ngates = run(n, fusion_k, None)
    greedy, b, _ = run(n, fusion_k, 0)
    always, c, _ = run(n, fusion_k, 1)
    assert always < greedy
    assert got == (always if searched else greedy)
    if a is not None:
        # an op moves the state by at most 6 eps of its norm, either way
        tol = 2 * 6 * 2.0 ** -24 * ngates
        assert np.linalg.norm(a - b) <= tol and np.linalg.norm(a - c) <= tol

"""Recorded sweeps carry the features of the programs as the planner ranks them:
a circuit of one-qubit gates without controls gives one op per gate and no
controls, whatever form the kernels run the ops in."""
import numpy as np
import pytest

from q1tsim_amd.gvs import GpuVectorState

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jit", [False, True])
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [14, 17])
def test_recorded_features(n, precision, jit):
    rng = np.random.Generator(np.random.PCG64(n))
    g = GpuVectorState(n, 1, precision)
    g.set_jit(jit)
    g.set_recording(True)
    gates = 0
    for _ in range(3):
        for q in range(n):
            for name in ("h", "rz", "rx", "ry"):
                g.apply_named(name, [q], [] if name == "h" else [float(rng.uniform(0.1, 3.0))])
                gates += 1
    g.flush()
    feat, tiles, ms = g.take_samples()
    g.close()
    assert len(feat) and np.all(ms > 0) and np.all(tiles == 1 << (n - 12))
    ops = feat[:, 3] + feat[:, 4] + feat[:, 5] + feat[:, 6]
    assert np.array_equal(ops, feat[:, 15])    # one op per gate
    assert not feat[:, 7:10].any()             # thread, register and outer controls
    assert feat[:, 15].sum() <= gates
    assert np.all(feat[:, 19] == (1 if jit else 0))

"""One-qubit marginals (items.hip): Z against the column's weights, X and Y
through the outcome counts of a peek with known uniforms.  Sizes: below and at
one workgroup's share (2^12 work units complex128, 2^13 complex64), around
256 workgroups per column, lowest / middle / highest qubit bit, several
columns of one state."""
import numpy as np
import pytest

from q1tsim_amd._lib import lib
from q1tsim_amd.gvs import GpuVectorState, Xoshiro

pytestmark = pytest.mark.gpu


def uniforms(seed, count):
    x = lib().q1t_xoshiro_new(seed)
    u = np.array([(lib().q1t_xoshiro_next(x) >> 12) * 2.0 ** -52 for _ in range(count)])
    lib().q1t_xoshiro_free(x)
    return u


def pairs(col, n, q):
    v = col.reshape(1 << q, 2, 1 << (n - 1 - q))
    return v[:, 0].ravel(), v[:, 1].ravel()


# a sum of m positive terms of total 1, each rounded once and added by trees
# and runs of at most 2^9 terms: relative error below 2^10 * 2^-53
TOL = 2.0 ** -43


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 7, 12, 13, 14, 15, 20, 21, 22])
def test_marginals(n, precision):
    shots = 257
    s = GpuVectorState(n, shots, precision)
    s.set_random_normal(100 + n)
    col = s.column(0)
    for q in sorted({0, n // 2, n - 1}):
        a0, a1 = pairs(col, n, q)
        w = float(np.sum(a0.real ** 2 + a0.imag ** 2))
        assert abs(s.marginal_w0(q)[0] - w) <= TOL
        assert np.array_equal(s.marginal_w0_noalloc(q), s.marginal_w0(q))
        for basis, b0 in (("X", a0 + a1), ("Y", a0 - 1j * a1)):
            w = 0.5 * float(np.sum(b0.real ** 2 + b0.imag ** 2))
            u = uniforms(7 * n + q, shots)
            assert np.min(np.abs(u - w)) > TOL      # no draw on the edge
            res = np.zeros(shots, np.uint64)
            s.measure_into(q, 0, res, Xoshiro(7 * n + q), collapse=False, basis=basis)
            assert int(np.sum(res == 0)) == int(np.sum(u < w))
    s.close()


def test_marginals_of_several_columns():
    n, shots = 14, 300
    s = GpuVectorState(n, shots, "c128")
    s.set_random_normal(3)
    res, rng = np.zeros(shots, np.uint64), Xoshiro(5)
    for q in (0, 6, 13):
        s.measure_into(q, q, res, rng)
    assert s.ncols > 4
    for q in (0, 3, 13):
        exp = [float(np.sum(np.abs(pairs(s.column(c), n, q)[0]) ** 2)) for c in range(s.ncols)]
        assert np.max(np.abs(s.marginal_w0(q) - exp)) <= TOL
        assert np.array_equal(s.marginal_w0_noalloc(q), s.marginal_w0(q))
    s.close()

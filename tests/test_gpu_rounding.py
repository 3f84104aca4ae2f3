"""The shared-part FP64 divisions and square roots of the step kernels over
the magnitudes a state can hold: the RHS against the oracle's plain divisions
and square roots.

Tolerance: each quotient and root is correctly rounded (0.5 / c to one ulp),
so a component differs by a few ulp of its largest face term; a mesh this
small has at most four faces per cell and depths within a factor of two, so
1e-13 of the component's largest value leaves a factor of 100.
"""
import numpy as np
import pytest

from hgswe import capi, cases
import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell_kernel", [False, True])
@pytest.mark.parametrize("depth", [2e-3, 1.0, 3e4])
@pytest.mark.parametrize("q", [1e-300, 1e-150, 1e-8, 1.0, 1e4])
def test_rhs_over_magnitudes(depth, q, cell_kernel):
    c = cases.dam_break(nx=13, ny=9, n=1e-6)
    rng = np.random.default_rng(3)
    N = c.N
    Q = np.concatenate([depth * rng.uniform(1.0, 2.0, N) if q >= 1e-8 else np.full(N, depth), q * rng.normal(size=2 * N)])
    r, ref = capi.Context(c, cell_kernel=cell_kernel).rhs(Q), pyoracle.Oracle(c).rhs(Q)
    assert np.all(np.isfinite(ref))
    for k in range(3):
        a, b = r[k * N:(k + 1) * N], ref[k * N:(k + 1) * N]
        assert np.max(np.abs(a - b)) <= 1e-13 * max(np.max(np.abs(b)), 1e-305), (k, np.max(np.abs(a - b)), np.max(np.abs(b)))


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_non_finite_state_is_reported(bad):
    c = cases.dam_break(nx=13, ny=9)
    for at in (5, c.N + 5, 2 * c.N + 5):
        Q = c.Q0.copy()
        Q[at] = bad
        with pytest.raises(capi.HGError) as e:
            capi.Context(c).step(Q, 1e-3, 3)
        assert e.value.code == capi.HG_ERR_NONFINITE

"""The block -> tile mapping that a mesh starts with: the steps, the gradient
and the RHS are those of the mapping of work-group b to tile b, bit for bit,
whatever number of tiles the windows leave over."""
import numpy as np
import pytest

from hgswe import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [2_500, 40_000, 132_000, 140_000, 150_000, 260_000])
def test_default_mapping_has_the_identity_mappings_bits(cells):
    c = cases.channel(cells, seed=9, nsteps=10)
    a, b = capi.Context(c), capi.Context(c)
    T, chunk = a.tile_config()
    b.set_tile_config(T, 0)
    print(f"  {c.N} cells, tiles of {T}, runs of {chunk}", flush=True)
    assert np.array_equal(a.rhs(c.Q0), b.rhs(c.Q0))
    assert np.array_equal(a.step(c.Q0, c.dt, 3), b.step(c.Q0, c.dt, 3))
    bar = np.random.default_rng(cells).normal(size=3 * c.N)
    for x, y in zip(a.adjoint(c.Q0, c.dt, 3, 0, bar), b.adjoint(c.Q0, c.dt, 3, 0, bar)):
        assert np.array_equal(x, y)

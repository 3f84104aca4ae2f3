"""Forward mode of a FlowResistance network with n as the active parameter: n
enters through the inlets (their conveyance and ghost states), the network
through the friction, and the two tangents are separate.  Checked against the
reverse mode: <lam, J dp> = <J^T lam, dp> for the state and n together."""
import numpy as np
import pytest

from hgswe import capi

from test_gpu_resident import channel, mixed, moving, with_law

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 256])
@pytest.mark.parametrize("name", ["channel", "mixed"])
def test_transpose_of_reverse_mode(name, tile):
    """12 steps of about 1,000 operations a cell, errors relative to the sum of the terms' magnitudes: 12 x 1000 x
    2^-53 = 1.3e-12 on either side."""
    c = moving(channel(1100) if name == "channel" else mixed(900, 2))
    rng = np.random.default_rng(7)
    ctx = capi.Context(c)
    if tile:
        ctx.set_tile_config(tile)
    with_law(ctx, c, "FlowResistance")
    lam, d0, dn = rng.normal(size=3 * c.N), rng.normal(size=3 * c.N), 1e-2 * rng.normal(size=c.N)
    Qb, nb, _, _ = ctx.adjoint(c.Q0, c.dt, 12, 0, lam)
    assert np.any(nb)
    ctx.set_active_param(capi.HG_PARAM_N_CELL)
    for a, b in ((d0, dn), (0.0 * d0, dn), (d0, 0.0 * dn)):
        dQ = ctx.jvp(c.Q0, c.dt, 12, dQ0=a, params=c.n, dparams=b)[1]
        lhs, rhs = lam @ dQ, Qb @ a + nb @ b
        size = np.abs(lam) @ np.abs(dQ) + np.abs(Qb) @ np.abs(a) + np.abs(nb) @ np.abs(b)
        assert abs(lhs - rhs) <= 2.6e-12 * size

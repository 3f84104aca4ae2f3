"""Host arrays that pass through a context's pinned block.

An array that fits the block is copied into it and moved by one kernel, with
no wait; a larger one goes through the process's chunked buffers.  Bitwise
round trips on both sides of the limit and at the edges of the chunks, more
uploads in a row than the block has room for, and the working copies of the
fields, which are written again only when something changed them.
"""
import numpy as np
import pytest

from hgswe import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [180, 5_000, 43_000, 47_000, 87_000, 88_500, 175_000])
def test_round_trips_are_bitwise(cells):
    c = cases.channel(cells, seed=3, nsteps=10)
    ctx = capi.Context(c)
    rng = np.random.default_rng(cells)
    print(f"  {c.N} cells", flush=True)
    for _ in range(3):
        qs = [rng.normal(size=3 * c.N) for _ in range(7)]  # the pieces of the block are used up in between
        for q in qs:
            ctx.upload(q)
            q_sent = q.copy()
            q[:] = np.nan  # the caller's array is its own again on return
        assert np.array_equal(ctx.download(), q_sent)
    want = capi.Context(c).rhs(c.Q0)
    for _ in range(3):
        assert np.array_equal(ctx.rhs(c.Q0), want)


@pytest.mark.parametrize("kind", ["n", "zb", "Q"])
def test_fields_come_back_after_a_parameter(kind):
    """RHS with the fields, with a parameter in their place, with the fields again."""
    c = cases.channel(2_000, seed=5, nsteps=10)
    ctx = capi.Context(c)
    base = ctx.rhs(c.Q0)
    p = {"n": np.array([0.05]), "zb": c.zb + 0.01 * np.cos(np.arange(c.N)), "Q": 1.25 * np.asarray(c.inletQ)}[kind]
    zone = np.zeros(c.N, dtype=np.int32) if kind == "n" else None
    ctx.set_active_param({"n": capi.HG_PARAM_N_ZONE, "zb": capi.HG_PARAM_ZB, "Q": capi.HG_PARAM_Q}[kind], zone, 1)
    with_p = ctx.rhs(c.Q0, p)
    assert not np.array_equal(with_p, base)
    assert np.array_equal(ctx.rhs(c.Q0, p), with_p)
    ctx.set_active_param(capi.HG_PARAM_NONE)
    assert np.array_equal(ctx.rhs(c.Q0), base)
    assert np.array_equal(ctx.rhs(c.Q0), base)

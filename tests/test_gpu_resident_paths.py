"""Which path a small mesh takes (resident runs or one launch per step) is a
matter of speed: changes of tiling, inputs that a resident run does not hold
and waits that run out leave the results as they are."""
import dataclasses

import numpy as np
import pytest

from hgswe import capi, cases
from hgswe import mesh as hm

from test_gpu_resident import LAWS, REVERSE, channel, moving, two_inlets, with_law

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("between", [("tile", 256), ("tile", 256, 128), ("tile", 512), ("adjoint", 256),
                                     ("adjoint", 256, 0), ("tune",)])
@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h"])
def test_tiled_anew_between_the_sweeps(law, between):
    """Between hg_adjoint_forward and hg_adjoint_reverse the mesh is tiled anew: the same cotangents (bit for bit with n
    from the field; the closures' bound is that of test_reverse_run_with_closure)."""
    c = moving(channel(1100))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ref, ctx = capi.Context(c), capi.Context(c)
    for k in (ref, ctx):
        with_law(k, c, law)
    want = ref.adjoint(c.Q0, c.dt, 12, 0, lam)
    if between[0] == "adjoint":  # the forward sweep under the other size
        ctx.set_adjoint_tile(between[1])
    QN = ctx.adjoint_forward(c.Q0, c.dt, 12, 0)
    assert np.array_equal(QN, ref.step(c.Q0, c.dt, 12))
    for size in between[1:]:
        (ctx.set_tile_config if between[0] == "tile" else ctx.set_adjoint_tile)(size)
    if between[0] == "tune":
        ctx.autotune(c.dt, 8)
    for x, y in zip(ctx.adjoint_reverse(lam), want):
        if law == "field":
            assert np.array_equal(x, y)
        else:
            assert np.max(np.abs(x - y), initial=0.0) <= 1.3e-11 * np.max(np.abs(y), initial=0.0)


@pytest.mark.parametrize("keep", [1, 20])
def test_inlet_faces_left_out_of_the_list(keep):
    """Ghosts of inlet kind that their inlet's list does not name read its conveyance without adding to it: the same
    bits with and without a tiling that runs resident."""
    c = two_inlets(8000)
    m = c.mesh
    lists = [m.inlet_ghost[m.inlet_off[b]:m.inlet_off[b + 1]] for b in range(m.n_inlet)]
    assert all(len(x) > 40 for x in lists)
    lists[0] = lists[0][:keep]
    c = dataclasses.replace(c, mesh=dataclasses.replace(
        m, inlet_off=np.array([0, keep, keep + len(lists[1])], dtype=np.int32), inlet_ghost=np.concatenate(lists)))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_tile_config(256)
    assert np.array_equal(ctx.step(c.Q0, c.dt, 30), single.step(c.Q0, c.dt, 30))
    for x, y in zip(ctx.adjoint(c.Q0, c.dt, 30, 0, lam), single.adjoint(c.Q0, c.dt, 30, 0, lam)):
        assert np.all(np.isfinite(y)) and np.array_equal(x, y)


def second_inlet_walled(c):
    """The case with the faces of its second inlet as walls: that inlet is left without faces."""
    m = c.mesh
    off = int(m.inlet_off[1])
    kind = m.ghost_kind.copy()
    kind[m.inlet_ghost[off:]] = hm.BC_WALL
    return dataclasses.replace(c, mesh=dataclasses.replace(
        m, ghost_kind=kind, inlet_off=np.array([0, off, off], dtype=np.int32), inlet_ghost=m.inlet_ghost[:off]))


@pytest.mark.parametrize("n", [30, 300, 2000])
def test_inlet_without_faces(n):
    """Its discharge enters nowhere: its cotangent is zero, and the others are the per-tile kernel's."""
    both = two_inlets(n)
    c = second_inlet_walled(both)
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    single = capi.Context(c)
    single.set_tile_config(256)
    want = single.adjoint(c.Q0, c.dt, 12, 0, lam)
    assert want[3][1] == 0.0
    for _ in range(3):  # contexts whose second inlet has a cotangent leave it in the memory that the next one takes
        used = capi.Context(both)
        assert used.adjoint(both.Q0, both.dt, 12, 0, lam)[3][1] != 0.0
        used.close()
        ctx = capi.Context(c)
        for x, y in zip(ctx.adjoint(c.Q0, c.dt, 12, 0, lam), want):
            assert np.array_equal(x, y)
        ctx.close()


@pytest.mark.parametrize("n", [300, 8000])
def test_roughness_cotangent_of_inlet_cells(n):
    """An inlet cell's n has a boundary and a friction term, which the two paths add at different places."""
    c = two_inlets(n)
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_tile_config(256)
    for seed in range(8):
        lam = np.random.default_rng(seed).normal(size=3 * c.N)
        for x, y in zip(ctx.adjoint(c.Q0, c.dt, 12, 0, lam), single.adjoint(c.Q0, c.dt, 12, 0, lam)):
            assert np.array_equal(x, y)


# ---- which path ran, and a wait that runs out
CALLS = {
    "step": lambda k, c, lam: [k.step(c.Q0, c.dt, 12)],
    "adjoint": lambda k, c, lam: list(k.adjoint(c.Q0, c.dt, 12, 0, lam)),
    "reverse": lambda k, c, lam: list(k.adjoint_reverse(lam)),
    "jvp": lambda k, c, lam: list(k.jvp(c.Q0, c.dt, 12, dQ0=lam)),
    "tsit5": lambda k, c, lam: [k.tsit5(c.Q0, 0.0, 12 * c.dt, 3, dt0=c.dt)[0]],
}


def resident_and_single(c, law, call, lam):
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_resident(capi.HG_RESIDENT_OFF)
    for k in (ctx, single):
        with_law(k, c, law)
        if call == "reverse":
            k.adjoint_forward(c.Q0, c.dt, 12, 0)
    return ctx, single


@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h"])
@pytest.mark.parametrize("call", sorted(CALLS))
def test_resident_runs_are_taken(call, law):
    c = moving(channel(1100))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ctx, single = resident_and_single(c, law, call, lam)
    before = ctx.resident()[1]
    CALLS[call](ctx, c, lam)
    CALLS[call](single, c, lam)
    assert ctx.resident() == (True, before + (2 if call == "adjoint" else 1), 0)
    assert single.resident() == (False, 0, 0)


@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h"])
@pytest.mark.parametrize("call", sorted(CALLS))
def test_a_wait_that_runs_out(call, law):
    """One tile is left out of the run and the others give up waiting for it (after a second); the call starts over with
    single launches."""
    c = moving(channel(1100))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ctx, single = resident_and_single(c, law, call, lam)
    want = CALLS[call](single, c, lam)
    if law != "field" and call in ("adjoint", "reverse"):
        want.append(single.lux_grad() if law == "ManningN_h" else want[0])
    before = ctx.resident()[1]
    ctx.set_resident(capi.HG_RESIDENT_SHORT)
    got = CALLS[call](ctx, c, lam)
    if law != "field" and call in ("adjoint", "reverse"):
        got.append(ctx.lux_grad() if law == "ManningN_h" else got[0])
    assert ctx.resident() == (False, before, 1)
    for x, y in zip(got, want):
        assert np.array_equal(x, y)
    ctx.set_resident(capi.HG_RESIDENT_ON)
    ctx.step(c.Q0, c.dt, 12)
    assert ctx.resident() == (True, before + 1, 1)
    with pytest.raises(capi.HGError):
        ctx.set_resident(4)


@pytest.mark.parametrize("n", [300, 1100, 9000, 40000, 98000])
def test_tuned_meshes_step_resident(n):
    """The tuner compares a resident run with the single launches, and leaves a mesh that it suits to it."""
    c = channel(n)
    ctx, ref = capi.Context(c), capi.Context(c)
    ctx.upload(c.Q0)
    T, x, ms = ctx.autotune(c.dt, 16)
    assert (T, x) == ctx.tile_config() and T == 128 and ms > 0.0
    assert np.array_equal(ctx.download(), c.Q0)
    runs = ctx.resident()[1]
    assert np.array_equal(ctx.step(c.Q0, c.dt, 40), ref.step(c.Q0, c.dt, 40))
    assert ctx.resident() == (True, runs + 1, 0)
    ctx.set_resident(capi.HG_RESIDENT_OFF)
    assert np.array_equal(ctx.step(c.Q0, c.dt, 40), ref.step(c.Q0, c.dt, 40))


@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h"])
@pytest.mark.parametrize("call", sorted(CALLS))
def test_no_memory_for_the_run(call, law):
    """Where a resident run's own memory (rings, sums, Tsit5's frames, a law's recorded n) is not to be had, the call
    takes single launches; with the memory it runs resident again."""
    c = moving(channel(1100))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_resident(capi.HG_RESIDENT_OFF)
    ctx.set_resident(capi.HG_RESIDENT_NOMEM)
    for k in (ctx, single):
        with_law(k, c, law)
        if call == "reverse":
            k.adjoint_forward(c.Q0, c.dt, 12, 0)
    for x, y in zip(CALLS[call](ctx, c, lam), CALLS[call](single, c, lam)):
        assert np.array_equal(x, y)
    assert ctx.resident() == (True, 0, 0)
    ctx.set_resident(capi.HG_RESIDENT_ON)
    assert np.array_equal(ctx.step(c.Q0, c.dt, 12), single.step(c.Q0, c.dt, 12))
    assert ctx.resident() == (True, 1, 0)


def test_reversal_without_memory_for_the_law():
    """The forward run is resident, its law's n of each step is not recorded: the reversal takes single launches."""
    c = moving(channel(1100))
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_resident(capi.HG_RESIDENT_OFF)
    for k in (ctx, single):
        with_law(k, c, "sigmoid")
    ctx.step(c.Q0, c.dt, 12)  # takes the ring
    ctx.set_resident(capi.HG_RESIDENT_NOMEM)
    for x, y in zip(ctx.adjoint(c.Q0, c.dt, 12, 0, lam), single.adjoint(c.Q0, c.dt, 12, 0, lam)):
        assert np.array_equal(x, y)
    assert ctx.resident() == (True, 2, 0)


# ---- the same bits from either path: the results do not depend on which one had room, memory or enough steps
@pytest.mark.parametrize("law", sorted(LAWS))
@pytest.mark.parametrize("name", sorted(REVERSE))
def test_forward_mode_has_the_same_bits(name, law):
    c = moving(REVERSE[name]()) if name != "wet_dry" else REVERSE[name]()
    if name == "wet_dry" and law == "h_Umag_ks":
        pytest.skip("the law has no value at rest")
    rng = np.random.default_rng(11)
    d0 = 1e-2 * rng.normal(size=3 * c.N)
    kinds = [capi.HG_PARAM_NONE, capi.HG_PARAM_ZB] + ([capi.HG_PARAM_Q] if c.mesh.n_inlet else [])
    kinds += [capi.HG_PARAM_N_CELL] if law in ("field", "FlowResistance") else []
    kinds += [capi.HG_PARAM_UDE] if LAWS[law] in (1, 2, 3) else []
    for kind in kinds:
        ctx, single = capi.Context(c), capi.Context(c)
        single.set_resident(capi.HG_RESIDENT_OFF)
        out = []
        for k in (ctx, single):
            w = with_law(k, c, law)
            k.set_active_param(kind)
            p = {capi.HG_PARAM_NONE: None, capi.HG_PARAM_ZB: c.zb, capi.HG_PARAM_N_CELL: c.n,
                 capi.HG_PARAM_Q: c.inletQ, capi.HG_PARAM_UDE: w}[kind]
            dp = None if p is None else np.random.default_rng(12).normal(size=np.size(p)) * 1e-3
            out.append(k.jvp(c.Q0, c.dt, 24, dQ0=d0, params=p, dparams=dp))
        for x, y in zip(*out):  # (the power law has no finite value on dry cells)
            assert np.any(np.isfinite(y)) and np.array_equal(x, y, equal_nan=True), kind


@pytest.mark.parametrize("law", ["sigmoid", "power_law", "h_Umag_ks", "ManningN_h", "ManningN_h_Umag_ks",
                                 "FlowResistance", "one_layer", "three_layers"])
@pytest.mark.parametrize("name", ["one_tile", "tile_and_one", "tiny_channel", "channel", "mixed", "two_inlets", "quads",
                                  "batch"])
def test_gradients_through_closures_have_the_same_bits(name, law):
    """Whole, by segments, and by single launches under another tiling: every cotangent, the weights' among them."""
    c = moving(REVERSE[name]())
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    out = []
    for mode, tile, kck in ((capi.HG_RESIDENT_ON, 128, 0), (capi.HG_RESIDENT_ON, 128, 5), (capi.HG_RESIDENT_OFF, 256, 3)):
        ctx = capi.Context(c)
        ctx.set_resident(mode)
        ctx.set_tile_config(tile)
        net = law in ("one_layer", "three_layers")
        if net:
            hidden, acts = ([4], ["sigmoid"]) if law == "one_layer" else ([3, 2, 4], ["tanh", "leakyrelu", "softplus"])
            n = capi.lux_net("ManningN_h", hidden, acts, (0.02, 0.06), (0.1, 4.0))
            ctx.set_lux_ude(n, 0.5 * np.random.default_rng(2).normal(size=capi.lux_n_params(n)))
        else:
            net = with_law(ctx, c, law) is not None
        out.append(list(ctx.adjoint(c.Q0, c.dt, 12, kck, lam)) + ([ctx.lux_grad()] if net else []))
        assert (ctx.resident()[1] > 0) == (mode == capi.HG_RESIDENT_ON)
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert np.all(np.isfinite(y)) and np.array_equal(x, y)


@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h", "FlowResistance"])
@pytest.mark.parametrize("name", ["one_tile", "tile_and_one", "quads", "tiny_channel", "channel", "mixed", "two_inlets",
                                  "two_inlets_large"])
def test_tsit5_has_the_same_bits(name, law):
    """The adaptive integrator takes the same steps: frames and counts, over a few steps and over several launches."""
    c = REVERSE[name]()
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_resident(capi.HG_RESIDENT_OFF)
    for k in (ctx, single):
        with_law(k, c, law)
    for T, frames, tol in ((12 * c.dt, 3, 1e-3), (60 * c.dt, 7, 1e-4)):
        (F, n), (G, m) = [k.tsit5(c.Q0, 0.0, T, frames, dt0=0.1 * c.dt, reltol=tol) for k in (ctx, single)]
        assert n == m and np.all(np.isfinite(G)) and np.array_equal(F, G)
    assert ctx.resident()[1] >= 2


def test_tsit5_has_the_same_bits_over_many_launches():
    c = cases.dam_break(nx=40, ny=5)
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_resident(capi.HG_RESIDENT_OFF)
    (F, n), (G, m) = [k.tsit5(c.Q0, 0.0, 120.0, 3, abstol=1e-13, reltol=1e-12, dt0=1e-3) for k in (ctx, single)]
    assert n == m and n[0] + n[1] > 1024 and np.array_equal(F, G)
    assert ctx.resident()[1] >= 2

"""Resident runs (many steps of a small mesh in one launch) against the
per-cell kernel, one launch per step, bit for bit: the two form every value
with the same operations in the same order, so the tolerance is zero.

Sizes around one tile of 128 cells and several tiles, triangles, quads and a
mix, closed domains and inlets (within one tile, over several, two on one
cell), wet / dry fronts, per-instance time steps, recorded runs, and contexts
on several threads that do not fit on the device together.
"""
import threading

import numpy as np
import pytest

from hgswe import capi, cases
from hgswe import mesh as hm

pytestmark = pytest.mark.gpu


def channel(n, seed=3, **kw):
    return cases.channel(n, seed=seed, Lx=max(30.0, 0.25 * n ** 0.5 * 10), Ly=max(6.0, 0.025 * n ** 0.5 * 10),
                         Q_in=2.0, n_bumps=2, **kw)


def mixed(n_quads, seed):
    nx = max(2, int(round((4.0 * n_quads) ** 0.5)))
    xy, quads, side = cases.rect_quads(10.0 * nx, 10.0 * max(1, n_quads // nx), nx, max(1, n_quads // nx))
    rng = np.random.default_rng(seed)
    cells = []
    for a, b, c, d in quads:
        cells += [[a, b, c, -1], [a, c, d, -1]] if rng.random() < 0.5 else [[a, b, c, d]]
    m = hm.build_mesh(xy, np.array(cells), {1: side["left"], 2: side["right"], 3: side["bottom"], 4: side["top"]},
                      {1: "INLET-Q", 2: "EXIT-H", 3: "WALL", 4: "SYMM"})
    zb = 0.2 * rng.random(m.n_cells)
    zg, S0x, S0y = hm.bed_data(m, zb)
    h = 2.0 + 0.2 * rng.random(m.n_cells)
    hs = np.full(m.n_cells, 0.3)
    c = cases.Case(name="mixed", mesh=m, hstill=hs, hstill_ghost=hs[m.ghost_cell], zb=zb, zb_ghost=zg, S0x=S0x, S0y=S0y,
                   n=rng.uniform(0.02, 0.05, m.n_cells), inletQ=np.array([3.0]), exitWSE=np.array([2.1]),
                   Q0=np.concatenate([h - hs, np.zeros(2 * m.n_cells)]), dt=0.0, nsteps=0)
    c.dt = cases.cfl_dt(c, 0.3)
    return c


def check(c, steps, ctx=None, dts=None):
    ctx, ref = ctx or capi.Context(c), capi.Context(c, cell_kernel=True)
    if dts is not None:
        ctx.batch_set_dt(dts)
        ref.batch_set_dt(dts)
    a, b = ctx.step(c.Q0, c.dt, steps), ref.step(c.Q0, c.dt, steps)
    assert np.all(np.isfinite(b)) and (c.N == 1 or not np.array_equal(b, c.Q0))
    assert np.array_equal(a, b)
    return ctx


@pytest.mark.parametrize("nx,ny", [(1, 1), (4, 3), (16, 8), (43, 3), (32, 4), (100, 10)])
@pytest.mark.parametrize("steps", [4, 5, 6, 7, 33])
def test_closed_quads(nx, ny, steps):
    check(cases.dam_break(nx=nx, ny=ny), steps)


@pytest.mark.parametrize("n", [40, 126, 260, 1100, 9000, 40000])
def test_channel_triangles(n):
    c = channel(n)
    ctx = check(c, 40)
    ctx.upload(c.Q0)  # in pieces: each run starts from the other state buffer
    for k in (7, 4, 3, 26):
        ctx.advance(c.dt, k)
    assert np.array_equal(ctx.download(), ctx.step(c.Q0, c.dt, 40))


@pytest.mark.parametrize("n", [30, 400, 3000])
def test_mixed_mesh(n):
    check(mixed(n, n), 30)


def test_no_renumbering():
    """Cells in a random order: tiles of up to three cross-tile faces per cell are run with one launch per step."""
    c = channel(800)
    check(c, 20, ctx=capi.Context(c, reorder=False))


def test_wet_dry_fronts():
    c = cases.channel(6_000, seed=12, Lx=1500.0, Ly=150.0, Q_in=60.0)
    x = c.mesh.centroid[:, 0]
    Q = c.Q0.copy()
    Q[:c.N] = np.where(x < 500.0, np.maximum(c.h_small, 2.2 - c.zb), c.h_small) - c.hstill
    check(c.copy_fields(Q0=Q, dt=cases.cfl_dt(c, 0.4, Q)), 60)


def test_batch_with_own_time_steps():
    parts = [channel(n, seed=n) for n in (90, 700, 300)]
    c = cases.concat(parts)
    check(c, 25, dts=[p.dt * f for p, f in zip(parts, (0.5, 0.8, 0.9))])
    check(c, 25)


@pytest.mark.parametrize("kck", [0, 20, 7])
def test_recorded_run(kck):
    """The gradient through a recorded resident run is the one through single launches."""
    c = channel(2500)
    probe = np.arange(0, c.N, 50, dtype=np.int32)
    target = (c.Q0[:c.N] + c.hstill + c.zb)[probe] + 0.01
    other = capi.Context(c)
    other.set_tile_config(256)  # not the resident tiling
    a = capi.Context(c).grad_probes(c.Q0, c.dt, 20, kck, probe, target)
    b = other.grad_probes(c.Q0, c.dt, 20, 5, probe, target)
    assert a[0] == b[0]
    for x, y in zip(a[1:], b[1:]):
        assert np.array_equal(x, y)


def test_errors_are_reported():
    c = channel(1100)
    Q = c.Q0.copy()
    Q[:c.N] = c.h_small - c.hstill  # a dry inlet has no conveyance
    with pytest.raises(capi.HGError) as e:
        capi.Context(c).step(Q, c.dt, 10)
    assert e.value.code == capi.HG_ERR_CONVEYANCE
    Q = c.Q0.copy()
    Q[c.N // 2] = np.nan
    ctx = capi.Context(c)
    with pytest.raises(capi.HGError) as e:
        ctx.step(Q, c.dt, 10)
    assert e.value.code == capi.HG_ERR_NONFINITE
    assert np.array_equal(ctx.step(c.Q0, c.dt, 10), capi.Context(c, cell_kernel=True).step(c.Q0, c.dt, 10))


def test_threads_share_the_device():
    """Three contexts on three threads, more tiles than the device holds at once: those that do not fit step with
    single launches, and every result is the one of a run alone."""
    c = channel(90_000)
    ref = capi.Context(c).step(c.Q0, c.dt, 60)
    out = [None] * 3

    def work(k):
        ctx = capi.Context(c)
        out[k] = [ctx.step(c.Q0, c.dt, 60) for _ in range(4)]

    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert all(np.array_equal(q, ref) for qs in out for q in qs)


def two_inlets(n_quads=300):
    """Two inlets on opposite ends of a closed channel (each over several tiles of a larger mesh)."""
    nx = max(4, int(round(n_quads ** 0.5)))
    xy, quads, side = cases.rect_quads(20.0 * nx, 20.0 * nx, nx, nx)
    m = hm.build_mesh(xy, quads, {1: side["left"], 2: side["right"], 3: side["bottom"], 4: side["top"]},
                      {1: "INLET-Q", 2: "INLET-Q", 3: "EXIT-H", 4: "WALL"})
    zb = 0.1 * np.random.default_rng(5).random(m.n_cells)
    zg, S0x, S0y = hm.bed_data(m, zb)
    hs = np.full(m.n_cells, 0.3)
    c = cases.Case(name="two_inlets", mesh=m, hstill=hs, hstill_ghost=hs[m.ghost_cell], zb=zb, zb_ghost=zg, S0x=S0x,
                   S0y=S0y, n=np.full(m.n_cells, 0.03), inletQ=np.array([20.0, 30.0]), exitWSE=np.array([2.0]),
                   Q0=np.concatenate([2.0 - zb - hs, np.zeros(2 * m.n_cells)]), dt=0.0, nsteps=0)
    c.dt = cases.cfl_dt(c, 0.3)
    return c


def wet_dry():
    c = cases.channel(6_000, seed=12, Lx=1500.0, Ly=150.0, Q_in=60.0)
    x = c.mesh.centroid[:, 0]
    Q = c.Q0.copy()
    Q[:c.N] = np.where(x < 500.0, np.maximum(c.h_small, 2.2 - c.zb), c.h_small) - c.hstill
    return c.copy_fields(Q0=Q, dt=cases.cfl_dt(c, 0.4, Q))


REVERSE = {"one_tile": lambda: cases.dam_break(nx=16, ny=8), "tile_and_one": lambda: cases.dam_break(nx=43, ny=3),
           "quads": lambda: cases.dam_break(nx=100, ny=10), "tiny_channel": lambda: channel(40),
           "channel": lambda: channel(9000), "mixed": lambda: mixed(900, 2), "wet_dry": wet_dry,
           "two_inlets": two_inlets, "two_inlets_large": lambda: two_inlets(8000),
           "batch": lambda: cases.concat([channel(n, seed=n) for n in (90, 700, 300)])}


@pytest.mark.parametrize("name", sorted(REVERSE))
@pytest.mark.parametrize("steps", [4, 5, 30])
def test_reverse_run(name, steps):
    """The reverse sweep in one launch against one launch per step (another tile size), every cotangent, bit for bit."""
    c = REVERSE[name]()
    single = capi.Context(c)
    single.set_tile_config(256)
    ctx = capi.Context(c)
    lam = np.random.default_rng(steps).normal(size=3 * c.N)
    a, b = ctx.adjoint(c.Q0, c.dt, steps, 0, lam), single.adjoint(c.Q0, c.dt, steps, 0, lam)
    assert np.all(np.isfinite(b[0])) and np.any(b[1])
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    for wrt in (("n",), ("zb",), ("Q",), ()):  # the sums nobody asks for are left out
        QN = ctx.adjoint_forward(c.Q0, c.dt, steps, 0)
        assert np.array_equal(QN, single.step(c.Q0, c.dt, steps))
        got = ctx.adjoint_reverse(lam, wrt=wrt)
        assert np.array_equal(got[0], b[0])
        for k, w in enumerate(("n", "zb", "Q")):
            assert got[k + 1] is None if w not in wrt else np.array_equal(got[k + 1], b[k + 1])


def test_reverse_run_with_own_time_steps():
    parts = [channel(n, seed=n) for n in (90, 700, 300)]
    c = cases.concat(parts)
    out = []
    for size in (0, 256):
        ctx = capi.Context(c)
        if size:
            ctx.set_tile_config(size)
        ctx.batch_set_dt([p.dt * f for p, f in zip(parts, (0.5, 0.8, 0.9))])
        out.append(ctx.adjoint(c.Q0, c.dt, 12, 0, np.linspace(-1, 1, 3 * c.N)))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


# ---- forward mode, laws and networks, and Tsit5 ----
LAWS = {"field": None, "sigmoid": dict(kind="sigmoid", n_lower=0.02, n_upper=0.06, k=2.0, h_mid=1.5),
        "power_law": dict(kind="power_law", n_lower=0.02, n_upper=0.05, k=0.4),
        "h_Umag_ks": dict(kind="h_Umag_ks"), "ManningN_h": 1, "ManningN_h_Umag_ks": 3, "FlowResistance": 2}


def moving(c):
    """The case with water moving everywhere (the h_Umag_ks law has no value at rest)."""
    Q = c.Q0.copy()
    Q[c.N:] = 0.1 * np.random.default_rng(8).uniform(0.5, 1.5, 2 * c.N)
    return c.copy_fields(Q0=Q)


def with_law(ctx, c, law, seed=4):
    """Turns the named law or network on; returns the network's weights (None for a law)."""
    rng = np.random.default_rng(seed)
    ks = rng.uniform(0.02, 0.1, c.N)
    spec = LAWS[law]
    if spec is None:
        return None
    if isinstance(spec, dict):
        ctx.set_n_law(**spec, ks=ks if law == "h_Umag_ks" else None)
        return None
    bounds = (1e-3, 1e-2) if law == "FlowResistance" else (0.02, 0.06)
    net = capi.lux_net(law, [3, 4], ["tanh", "softplus"], bounds, (0.1, 4.0), (0.0, 2.0), (0.0, 0.2))
    w = 0.5 * rng.normal(size=capi.lux_n_params(net))
    ctx.set_lux_ude(net, w, ks=ks if law == "ManningN_h_Umag_ks" else None)
    return w


@pytest.mark.parametrize("law", sorted(LAWS))
@pytest.mark.parametrize("name", ["tiny_channel", "channel", "mixed", "two_inlets", "quads"])
def test_state_dependent_roughness(name, law):
    c = moving(REVERSE[name]())
    ctx, single = capi.Context(c), capi.Context(c)
    single.set_tile_config(256)
    for k in (ctx, single):
        with_law(k, c, law)
    for steps in (4, 21):
        assert np.array_equal(ctx.step(c.Q0, c.dt, steps), single.step(c.Q0, c.dt, steps))


@pytest.mark.parametrize("law", ["field", "sigmoid", "h_Umag_ks", "ManningN_h", "FlowResistance"])
@pytest.mark.parametrize("name", sorted(REVERSE))
def test_forward_mode(name, law):
    """Value: the step's bits.  Tangent: the per-cell dual kernel's, which sums a cell's faces in the same order and
    forms them with the same operations; the compiler may pick the two sides' sums differently, so a few ulp of the
    largest tangent per step: 24 steps x 100 operations x 2^-53 is 3e-13."""
    c = moving(REVERSE[name]()) if name != "wet_dry" else REVERSE[name]()
    if name == "wet_dry" and law == "h_Umag_ks":
        pytest.skip("the law has no value at rest")
    kinds = [capi.HG_PARAM_NONE, capi.HG_PARAM_ZB]
    if law == "field":
        kinds += [capi.HG_PARAM_N_CELL] + ([capi.HG_PARAM_Q] if c.mesh.n_inlet else [])
    if law in ("ManningN_h", "FlowResistance"):
        kinds += [capi.HG_PARAM_UDE]
    rng = np.random.default_rng(11)
    d0 = 1e-2 * rng.normal(size=3 * c.N)
    for kind in kinds:
        out = []
        for size in (0, 256):
            ctx = capi.Context(c)
            if size:
                ctx.set_tile_config(size)
            w = with_law(ctx, c, law)
            ctx.set_active_param(kind)
            p = {capi.HG_PARAM_NONE: None, capi.HG_PARAM_ZB: c.zb, capi.HG_PARAM_N_CELL: c.n,
                 capi.HG_PARAM_Q: c.inletQ, capi.HG_PARAM_UDE: w}[kind]
            dp = None if p is None else np.random.default_rng(12).normal(size=np.size(p)) * 1e-3
            out.append(ctx.jvp(c.Q0, c.dt, 24, dQ0=d0, params=p, dparams=dp))
            assert np.array_equal(out[-1][0], ctx.step(c.Q0, c.dt, 24, params=p))
        (Q, dQ), (R, dR) = out
        assert np.array_equal(Q, R)
        assert np.all(np.isfinite(dR)) and np.max(np.abs(dQ - dR)) <= 3e-13 * np.max(np.abs(dR)), kind


@pytest.mark.parametrize("law", ["field", "sigmoid", "ManningN_h"])
@pytest.mark.parametrize("name", ["one_tile", "tile_and_one", "quads", "channel", "mixed", "two_inlets"])
def test_tsit5(name, law):
    """The error norm's sum over the cells is grouped by tiles, so the step sizes differ by a few ulp from those of
    single launches; how far that carries depends on the flow, so the bound is measured: ten times what a change of
    the first step by two ulp does to the single-launch run itself (or 1e-13).  Over a short run most steps are set
    by the frames, not the error: 1e-13.  (FlowResistance friction is stiff at rest: its step sizes sit at the
    stability limit and no run of it is stable under such a change; its RHS is the Euler runs' above.)"""
    c = REVERSE[name]()
    T = 60 * cases.cfl_dt(c, 0.4)

    def run(size, T, first):
        ctx = capi.Context(c)
        if size:
            ctx.set_tile_config(size)
        with_law(ctx, c, law)
        return ctx.tsit5(c.Q0, 0.0, T, 7, dt0=0.01 * T * first, reltol=1e-4)

    short = 0.2 * T
    (F, n), (G, m) = run(0, short, 1.0), run(256, short, 1.0)
    assert n == m and n[0] >= 7
    assert np.array_equal(F[0], c.Q0)
    assert np.max(np.abs(F - G)) <= 1e-13 * np.max(np.abs(G))
    (F, n), (G, m), (H, k) = run(0, T, 1.0), run(256, T, 1.0), run(256, T, 1.0 + 2.0 ** -51)
    assert n == m or m != k
    for f, g, h in zip(F, G, H):
        assert np.max(np.abs(f - g)) <= max(1e-13 * np.max(np.abs(G)), 10 * np.max(np.abs(h - g)))


def test_tsit5_many_steps():
    """More trial steps than one launch takes, and the errors of the single-launch path."""
    c = cases.dam_break(nx=40, ny=5)
    a, b = capi.Context(c), capi.Context(c)
    b.set_tile_config(256)
    T = 120.0
    (F, n), (G, m) = [x.tsit5(c.Q0, 0.0, T, 3, abstol=1e-13, reltol=1e-12, dt0=1e-3) for x in (a, b)]
    assert n[0] + n[1] > 1024 and m[0] + m[1] > 1024
    assert np.max(np.abs(F - G)) <= 1e-9 * np.max(np.abs(G))  # both are within 1e-11 of the solution
    Q = c.Q0.copy()
    Q[3] = np.nan
    for ctx in (a, b):
        with pytest.raises(capi.HGError) as e:
            ctx.tsit5(Q, 0.0, 1.0, 2)
        assert e.value.code == capi.HG_ERR_NONFINITE
        assert np.array_equal(ctx.tsit5(c.Q0, 0.0, 1.0, 2)[0][0], c.Q0)


@pytest.mark.parametrize("law", ["sigmoid", "power_law", "h_Umag_ks", "ManningN_h", "ManningN_h_Umag_ks",
                                 "FlowResistance", "one_layer", "three_layers"])
@pytest.mark.parametrize("name", ["tiny_channel", "channel", "mixed", "two_inlets", "quads", "batch"])
def test_reverse_run_with_closure(name, law):
    """Every cotangent, those of the network's weights among them, against single launches.  The closure's
    derivatives are formed once per step and scaled, and the weight sums are grouped by tiles: 12 steps of about 1,000
    operations give 12 x 1000 x 2^-53 = 1.3e-12 of the largest component, times ten for sums of both signs.  (A network
    of three hidden layers is not held resident in reverse: its forward run is, and feeds the single launches.)"""
    c = moving(REVERSE[name]())
    lam = np.random.default_rng(1).normal(size=3 * c.N)
    out = []
    for size in (0, 256):
        ctx = capi.Context(c)
        if size:
            ctx.set_tile_config(size)
        net = law in ("one_layer", "three_layers")
        if net:
            hidden, acts = ([4], ["sigmoid"]) if law == "one_layer" else ([3, 2, 4], ["tanh", "leakyrelu", "softplus"])
            n = capi.lux_net("ManningN_h", hidden, acts, (0.02, 0.06), (0.1, 4.0))
            ctx.set_lux_ude(n, 0.5 * np.random.default_rng(2).normal(size=capi.lux_n_params(n)))
        else:
            net = with_law(ctx, c, law) is not None
        out.append(list(ctx.adjoint(c.Q0, c.dt, 12, 0, lam)) + ([ctx.lux_grad()] if net else []))
    for x, y in zip(*out):
        assert np.all(np.isfinite(y))
        assert np.max(np.abs(x - y), initial=0.0) <= 1.3e-11 * np.max(np.abs(y), initial=0.0)

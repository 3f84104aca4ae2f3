"""Performance cases: calls that programs make of the shallow-water library
through its Python binding (``hgswe.capi.Context``), from one right-hand side
on a thousand cells to the gradient of a run over a million.

A case is a dict of plain values:

  path     which call (see CASES below)
  mesh     "triangles" (jittered Delaunay), "quads", or "mixed" (quads, half
           of them split into two triangles), about `cells` cells of 10 m^2
           in a 10 : 1 rectangle
  water    "channel" (inlet discharge, outlet stage, a wavy surface over a
           bumpy bed), "dam_break" (walls, flat bed) or "release" (walls,
           water let go over a dry bumpy bed: wet / dry fronts)
  steps    explicit Euler steps of the call (CFL 0.4; 0.3 with dry fronts)

and what the path adds to that.  Meshes and beds depend on the case alone;
the flow, the roughness, discharges, network weights and probes come from the
seed.  ``exact`` states the same equations in plain torch, float64.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hydrograd.jl_amd"))

from hgswe import capi, cases, ude  # noqa: E402
from hgswe import mesh as hm  # noqa: E402

G, H_SMALL, EPS = 9.81, 1e-3, 2.0 ** -52
WALL, INLET, EXIT = hm.BC_WALL, hm.BC_INLETQ, hm.BC_EXITH

CASES = [
    # one RHS per call with host arrays, as an integrator outside the library asks for it: the smallest call ...
    dict(name="rhs_dam_break_1k", path="rhs", mesh="quads", cells=1000, water="dam_break"),
    # ... and the largest mesh of the benchmark
    dict(name="rhs_channel_1m", path="rhs", mesh="triangles", cells=1_000_000, water="channel"),
    # a forward run from a host state to a host state: the 1,000-cell dam break of the smoke test ...
    dict(name="step_dam_break_1k", path="step", mesh="quads", cells=1000, water="dam_break", steps=200),
    # ... and the benchmark's 1,000 steps on a million triangles
    dict(name="step_channel_1m", path="step", mesh="triangles", cells=1_000_000, water="channel", steps=1000),
    # a batch of independent catchments of different sizes, with wet / dry fronts, advanced together
    dict(name="step_batch_release", path="batch", mesh="triangles", cells=100_000, water="release", steps=200,
         instances=8),
    # the loop body of a parameter inversion: forward sweep, a loss of the caller's own, reverse sweep, on a mesh of
    # the size of a field site (zone roughness and inlet discharge)
    dict(name="inversion_mixed_1k", path="inversion", mesh="mixed", cells=1300, water="channel", steps=300),
    # the probe-misfit gradient with respect to a roughness per cell
    dict(name="gradient_channel_100k", path="gradient", mesh="triangles", cells=100_000, water="channel", steps=1000,
         wrt="n", probes=200),
    # the same with respect to roughness, bed and discharge on a million triangles
    dict(name="gradient_channel_1m", path="gradient", mesh="triangles", cells=1_000_000, water="channel", steps=200,
         wrt="n zb Q", probes=200),
    # an ensemble of weight sets of the roughness closure on one mesh: every set's weight gradient in one sweep
    dict(name="closure_fields_32", path="closure", mesh="triangles", cells=50_000, water="channel", steps=100,
         fields=32, probes=200),
    # one training iteration of the small roughness network on a one-dimensional channel
    dict(name="network_quads_200", path="network", mesh="quads", cells=200, water="channel", steps=1000),
    # the adaptive integrator with a depth-dependent roughness law, saving frames
    dict(name="tsit5_mixed_1k", path="tsit5", mesh="mixed", cells=1300, water="channel", steps=400, frames=20),
    # forward-mode sensitivity of a run to the zone roughness
    dict(name="tangent_mixed_1k", path="tangent", mesh="mixed", cells=1300, water="channel", steps=300),
]


def listed():
    return [dict(c) for c in CASES]


def draw(rng):
    """Another case: any path, sizes spread over the logarithm of the range that the listed cases of that path span
    (fewer steps on larger meshes)."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["rhs", "step", "batch", "inversion", "gradient", "closure", "network", "tsit5", "tangent"])
    mesh = rng.choice(["triangles", "quads", "mixed"])
    if path == "rhs":
        return dict(path=path, mesh=mesh, cells=log(300, 900_000), water=rng.choice(["channel", "dam_break", "release"]))
    if path == "step":
        cells = log(300, 900_000)
        return dict(path=path, mesh=mesh, cells=cells, water=rng.choice(["channel", "dam_break", "release"]),
                    steps=log(20, min(1000, 300_000_000 // cells)))
    if path == "batch":
        return dict(path=path, mesh="triangles", cells=log(10_000, 400_000), water=rng.choice(["channel", "release"]),
                    steps=log(20, 300), instances=rng.randint(2, 16))
    if path == "inversion":
        return dict(path=path, mesh=mesh, cells=log(300, 30_000), water="channel", steps=log(50, 400))
    if path == "gradient":
        cells = log(2000, 800_000)
        return dict(path=path, mesh="triangles", cells=cells, water="channel",
                    steps=log(20, min(1000, 100_000_000 // cells)), wrt=rng.choice(["n", "zb", "Q", "n zb Q"]),
                    probes=log(10, 500))
    if path == "closure":
        fields = rng.randint(1, 32)
        return dict(path=path, mesh="triangles", cells=log(2000, 40_000), water="channel", steps=log(20, 100),
                    fields=fields, probes=log(10, 200))
    if path == "network":
        return dict(path=path, mesh=mesh, cells=log(150, 5000), water="channel", steps=log(50, 800))
    if path == "tsit5":
        return dict(path=path, mesh=mesh, cells=log(300, 100_000), water="channel", steps=log(50, 400),
                    frames=rng.randint(1, 30))
    return dict(path=path, mesh=mesh, cells=log(300, 100_000), water="channel", steps=log(50, 400))


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=20)
def _terrain(mesh, cells, walls):
    """(mesh, bed elevation per cell, length, width) of a case: the site, the same for every seed."""
    Lx = math.sqrt(100.0 * cells)
    Ly = Lx / 10.0
    rng = np.random.default_rng(cells)
    if mesh == "triangles":
        nx = max(3, round(math.sqrt(5.0 * cells)))
        xy, nodes, side = cases.jittered_delaunay(nx, max(3, round(cells / 2.0 / nx)), Lx, Ly, seed=cells)
    else:
        quads = cells if mesh == "quads" else cells / 1.5
        nx = max(2, round(math.sqrt(10.0 * quads)))
        xy, nodes, side = cases.rect_quads(Lx, Ly, nx, max(2, round(quads / nx)))
        if mesh == "mixed":
            cut = rng.random(len(nodes)) < 0.5
            a, b, c, d = nodes.T
            none = np.full(len(nodes), -1)
            parts = np.stack([np.stack([a, b, c, np.where(cut, none, d)], 1), np.stack([a, c, d, none], 1)], 1)
            nodes = parts.reshape(-1, 4)[np.stack([np.ones_like(cut), cut], 1).ravel()]
    ends = ("WALL", "WALL") if walls else ("INLET-Q", "EXIT-H")
    m = hm.build_mesh(xy, nodes, {1: side["left"], 2: side["right"], 3: side["bottom"], 4: side["top"]},
                      {1: ends[0], 2: ends[1], 3: "WALL", 4: "WALL"})
    z = 1e-4 * (Lx - xy[:, 0])
    for _ in range(20):
        amp, w, cx, cy = rng.uniform(0, 0.5), Lx * rng.uniform(0.005, 0.03), rng.uniform(0, Lx), rng.uniform(0, Ly)
        z = z + amp * np.exp(-((xy[:, 0] - cx) ** 2 + (xy[:, 1] - cy) ** 2) / (2 * w * w))
    return m, hm.nodes_to_cells(m, z), Lx, Ly


def _case(mesh, cells, water, rng):
    """The library's case bundle: a site with the seed's flow and roughness."""
    m, bed, Lx, Ly = _terrain(mesh, cells, water != "channel")
    N, x, y = m.n_cells, m.centroid[:, 0], m.centroid[:, 1]
    zb = np.zeros(N) if water == "dam_break" else bed
    still = 0.0 if water == "release" else 0.2  # depth below the still-water level
    qx = qy = np.zeros(N)
    if water == "channel":
        h = 3.0 - zb
        for _ in range(4):  # long waves of up to 10 cm
            kx, ky, ph = rng.uniform(2, 30) / Lx, rng.uniform(1, 5) / Ly, rng.uniform(0, 6.28)
            h = h + rng.uniform(0, 0.1) * np.sin(kx * x + ph) * np.cos(ky * y)
        qx, qy = h * rng.uniform(0.1, 0.3), h * 0.02 * np.sin(6.28 * x / Lx + rng.uniform(0, 6.28))
    elif water == "dam_break":
        h = np.where(x < Lx / 2, rng.uniform(0.9, 1.1), rng.uniform(0.45, 0.55))
    else:
        h = np.where(x < Lx * rng.uniform(0.25, 0.4), np.maximum(2 * H_SMALL, rng.uniform(2.0, 2.4) - zb), 2 * H_SMALL)
    zone = np.minimum((5 * x / Lx).astype(np.int32), 4)
    zone_n = rng.uniform(0.02, 0.06, 5)
    zb_ghost, S0x, S0y = hm.bed_data(m, zb)
    hs = np.full(N, still)
    c = cases.Case(name=water, mesh=m, hstill=hs, hstill_ghost=hs[m.ghost_cell].copy(), zb=zb, zb_ghost=zb_ghost,
                   S0x=S0x, S0y=S0y, n=zone_n[zone], inletQ=np.full(m.n_inlet, 0.5 * Ly * rng.uniform(0.8, 1.2)),
                   exitWSE=np.full(m.n_exit, 3.0), Q0=np.concatenate([h - still, qx, qy]), dt=0.0, nsteps=0, zone=zone,
                   zone_n=zone_n, g=G, k_n=1.0, h_small=H_SMALL)
    c.dt = cases.cfl_dt(c, 0.3 if water == "release" else 0.4)
    return c


NET = dict(hidden=[3, 3], activations=["tanh", "tanh"], output_bounds=(0.03, 0.06), h_bounds=(0.1, 5.0))


def _inputs(case, seed):
    """Everything a case's call reads, as host arrays."""
    rng = np.random.default_rng(seed)
    path = case["path"]
    if path == "batch":
        sizes = np.random.default_rng(case["cells"]).lognormal(0.0, 0.8, case["instances"])
        sizes = np.maximum(500, sizes / sizes.sum() * case["cells"]).astype(int)
        c = cases.concat([_case(case["mesh"], int(k), case["water"], rng) for k in sizes])
    else:
        c = _case(case["mesh"], case["cells"], case["water"], rng)
        if path == "closure":
            c = cases.concat([c] * case["fields"])
    d = dict(case=c, N=c.N, dt=c.dt, steps=case.get("steps", 0))
    if path in ("gradient", "closure"):
        site = c.extra["instances"][0] if path == "closure" else c
        probe = rng.choice(site.N, size=min(case["probes"], site.N // 2), replace=False)
        wse = np.tile((site.Q0[:site.N] + site.hstill + site.zb)[probe], case.get("fields", 1))
        d["probe"] = np.concatenate([probe + k * site.N for k in range(case.get("fields", 1))]).astype(np.int32)
        d["target"] = wse + 0.05 * rng.normal(size=wse.size)
    if path == "gradient":
        d["n"] = 0.03 * np.exp(0.2 * rng.normal(size=c.N))
    if path == "closure":
        d["weights"] = np.stack([ude.xavier_weights(seed=int(s)) for s in rng.integers(1 << 30, size=case["fields"])])
    if path in ("inversion", "network"):
        d["target"] = c.Q0 + 0.02 * rng.normal(size=3 * c.N)
    if path == "network":  # Glorot-uniform layers, LayerNorm scale 1 and shift 0
        u = lambda a, b: rng.uniform(-1, 1, a * b) * math.sqrt(6.0 / (a + b))  # noqa: E731
        norm = [np.zeros(3), np.ones(3), np.zeros(3)]
        d["weights"] = np.concatenate([u(1, 3), *norm, u(3, 3), *norm, u(3, 1), np.zeros(1)])
    if path == "tsit5":
        d["law"] = dict(n_lower=0.02, n_upper=rng.uniform(0.05, 0.07), k=rng.uniform(1.0, 3.0), h_mid=rng.uniform(1.5, 2.5))
    if path == "tangent":
        d["dn"] = rng.normal(size=5) * 0.01
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    path, c = case["path"], d["case"]
    ctx = capi.Context(c, share_mesh=path == "closure")
    if path == "inversion" or path == "tangent":
        ctx.set_active_param(capi.HG_PARAM_N_ZONE, zone=c.zone, n_zones=5)
    if path == "gradient":
        ctx.set_active_param(capi.HG_PARAM_N_CELL)
    if path == "closure":
        ctx.set_ude(d["weights"], set_of_cell=np.repeat(np.arange(case["fields"]), c.N // case["fields"]))
    if path == "network":
        ctx.set_lux_ude(capi.lux_net("ManningN_h", **NET), d["weights"])
        ctx.set_active_param(capi.HG_PARAM_UDE)
    if path == "tsit5":
        ctx.set_n_law("sigmoid", **d["law"])
    d.update(ctx=ctx, path=path, wrt=tuple(case.get("wrt", "").split()), frames=case.get("frames", 0))
    return d


def run(s):
    ctx, c, path, dt, steps = s["ctx"], s["case"], s["path"], s["dt"], s["steps"]
    if path == "rhs":
        return ctx.rhs(c.Q0)
    if path in ("step", "batch"):
        return ctx.step(c.Q0, dt, steps)
    if path == "inversion":
        QN = ctx.adjoint_forward(c.Q0, dt, steps, 0, params=c.zone_n)
        Q0_bar, n_bar, _, inlet_bar = ctx.adjoint_reverse((QN - s["target"]) / s["N"], wrt=("n", "Q"))
        return QN, Q0_bar, np.bincount(c.zone, weights=n_bar, minlength=5), inlet_bar
    if path == "gradient":
        out = ctx.grad_probes(c.Q0, dt, steps, 0, s["probe"], s["target"], params=s["n"], wrt=s["wrt"])
        return [v for v in out if v is not None]
    if path == "closure":
        loss, _, _, inlet_bar = ctx.grad_probes(c.Q0, dt, steps, 0, s["probe"], s["target"], wrt=("Q",))
        return loss, inlet_bar, ctx.ude_grad()
    if path == "network":
        QN = ctx.adjoint_forward(c.Q0, dt, steps, 0, params=s["weights"])
        Q0_bar, _, _, _ = ctx.adjoint_reverse((QN - s["target"]) / s["N"], wrt=())
        return QN, Q0_bar, ctx.lux_grad()
    if path == "tsit5":
        frames, counts = ctx.tsit5(c.Q0, 0.0, dt * steps, s["frames"], dt0=dt)
        return frames, np.array(counts)
    return ctx.jvp(c.Q0, dt, steps, params=c.zone_n, dparams=s["dn"])


def work(case):
    """Bytes: every step has to read the cell's state and six constants and each of its faces (neighbour, normal,
    length), and write the state; a reverse step reads those, the cotangent and the recorded state and writes the
    cotangent and its parameters' sums; a host call moves its arrays once.  Operations: about 110 a face (each face
    once) and 60 a cell; three times that backward; a tangent doubles them; the closure's network has 353 weights."""
    deg = {"triangles": 3.0, "quads": 4.0, "mixed": 10.0 / 3.0}[case["mesh"]]
    cells = case["cells"] * case.get("fields", 1)
    mesh = (16 + 28 * deg + 24) * (1.0 / case.get("fields", 1)) + 8
    fwd, ops = 48 + mesh, 55 * deg + 60
    host = 48.0 * cells
    steps, path = case.get("steps", 1), case["path"]
    if path in ("inversion", "gradient", "closure", "network"):
        rev = 72 + mesh + 16
        net = {"closure": 4 * 353 * 2, "network": 4 * 25 * 4}.get(path, 0)
        return {"bytes": cells * steps * (fwd + rev) + host, "flops": cells * steps * (4 * ops + 3 * net)}
    if path == "tangent":
        return {"bytes": cells * steps * (fwd + 48) + 2 * host, "flops": cells * steps * 3 * ops}
    if path == "tsit5":  # six evaluations a step, each of about five Euler steps' length
        return {"bytes": cells * steps * 6 / 5 * fwd + 24.0 * cells * case["frames"], "flops": cells * steps * 6 / 5 * ops}
    return {"bytes": cells * steps * fwd + host, "flops": cells * steps * ops}


# ------------------------------------------------------- the same in torch --
class _Flow:
    """swe_2d_rhs and its Euler step in plain torch float64: arrays (fields, faces per cell, cells)."""

    def __init__(self, c, K=1):
        site = c.extra["instances"][0] if K > 1 else c
        m = site.mesh
        self.N, self.K = m.n_cells, K
        self.dev = "cuda" if torch.cuda.is_available() and self.N * K > 8000 else "cpu"
        t = lambda v, kind=torch.float64: torch.as_tensor(np.ascontiguousarray(v)).to(self.dev, kind)  # noqa: E731
        off, deg = m.face_off[:-1].astype(np.int64), m.cell_deg
        slot = np.stack([np.where(k < deg, off + k, -1) for k in range(int(deg.max()))])
        pick = lambda v: np.where(slot >= 0, v[np.maximum(slot, 0)], 0)  # noqa: E731
        nbr = np.where(slot >= 0, m.face_nbr[np.maximum(slot, 0)], 0)
        ghost = np.where(nbr < 0, ~nbr, 0)
        kind = np.where(nbr < 0, m.ghost_kind[ghost], -1)
        bc = np.where(nbr < 0, m.ghost_bc[ghost], 0)
        self.own = torch.arange(self.N, device=self.dev).expand(len(slot), self.N)
        self.nbr = torch.where(t(nbr < 0, torch.bool), self.own, t(np.maximum(nbr, 0), torch.int64))
        self.inlet, self.exit, self.wall = (t(kind == k, torch.bool) for k in (INLET, EXIT, WALL))
        self.solid = t(kind >= 0, torch.bool)
        self.bc_in, self.bc_out = t(np.where(kind == INLET, bc, 0), torch.int64), t(np.where(kind == EXIT, bc, 0), torch.int64)
        self.nx, self.ny, self.len = t(pick(m.face_nx)), t(pick(m.face_ny)), t(pick(m.face_len))
        self.area, self.hs, self.zb = t(m.area), t(site.hstill), t(site.zb)
        self.S0 = (t(site.S0x), t(site.S0y))
        self.Qin, self.stage = t(c.inletQ).reshape(K, -1), t(c.exitWSE).reshape(K, -1)
        faces = m.inlet_ghost.astype(np.int64)
        self.in_cell, self.in_len = t(m.ghost_cell[faces], torch.int64), t(m.ghost_len[faces])
        self.in_bc = t(m.ghost_bc[faces], torch.int64)
        self.n_in = m.n_inlet
        self.n0 = t(c.n).reshape(K, -1)
        self.Q0 = t(c.Q0).reshape(3, K, -1).transpose(0, 1).contiguous()  # (K, 3, N)

    def bed_slope(self, zb):
        zf = torch.where(self.solid, zb[self.own], 0.5 * (zb[self.own] + zb[self.nbr]))
        return tuple(-(n * zf * self.len).sum(0) / self.area for n in (self.nx, self.ny))

    def rhs(self, Q, n, zb=None, S0=None, Qin=None):
        zb, S0, Qin = self.zb if zb is None else zb, S0 or self.S0, self.Qin if Qin is None else Qin
        xi = Q[:, 0]
        h = xi + self.hs
        wet = h > H_SMALL
        h, hu, hv = torch.where(wet, h, H_SMALL), torch.where(wet, Q[:, 1], 0.0), torch.where(wet, Q[:, 2], 0.0)
        nx, ny = self.nx, self.ny
        at = lambda v: v[..., self.nbr]  # noqa: E731
        L = [v[..., self.own] for v in (xi, h, hu, hv)]
        xR, hR, uR, vR = (at(v) for v in (xi, h, hu, hv))
        zL, zR = zb[self.own], zb[self.nbr]
        hsR = self.hs[self.nbr]
        # ghost cells: a wall mirrors the discharge; an inlet shares its discharge by conveyance; an outlet sets the stage
        uR, vR = torch.where(self.wall, -L[2], uR), torch.where(self.wall, -L[3], vR)
        if self.n_in:
            conv = torch.where(wet, h, 0.0)[:, self.in_cell] * self.in_len ** (5.0 / 3.0) / n[:, self.in_cell]
            total = torch.zeros_like(Qin).index_add(1, self.in_bc, conv)
            v = (Qin / total)[:, self.bc_in] * self.len ** (2.0 / 3.0) / n[..., self.own] * L[1] * wet[..., self.own]
            uR, vR = torch.where(self.inlet, -v * nx, uR), torch.where(self.inlet, -v * ny, vR)
        if self.stage.numel():
            hx = self.stage[:, self.bc_out] - zL
            hR = torch.where(self.exit, torch.where(hx > H_SMALL, hx, H_SMALL), hR)
        xR = torch.where(self.solid, hR - hsR, xR)
        f = self.flux(L[0], self.hs[self.own], L[1], L[2], L[3], zL, xR, hsR, hR, uR, vR, zR)
        d = [-(v * self.len).sum(1) / self.area for v in f]
        fr = G * n * n / (h + H_SMALL) ** (7.0 / 3.0) * torch.sqrt(hu * hu + hv * hv + EPS)
        src = [G * xi * s - fr * q for s, q in zip(S0, (hu, hv))]
        return torch.stack([d[0]] + [e + torch.where(wet, s, 0.0) for e, s in zip(d[1:], src)], 1)

    def flux(self, xL, sL, hL, uL, vL, zL, xR, sR, hR, uR, vR, zR):
        """Roe's flux with pre-balanced pressure; dry sides mirror the wet one below a step, or give its flux alone."""
        nx, ny = self.nx, self.ny
        dL, dR = hL <= H_SMALL, hR <= H_SMALL
        mR = dR & ~dL & (hL + zL < zR + H_SMALL)
        mL = dL & ~dR & (hR + zR < zL + H_SMALL)
        one = (dL ^ dR) & ~mL & ~mR
        h, u, v = torch.where(dL, hR, hL), torch.where(dL, uR, uL), torch.where(dL, vR, vL)  # the wet side
        p = 0.5 * G * (h + EPS) ** 2
        un = (u * nx + v * ny) / h
        alone = (un * h, un * u + p * nx, un * v + p * ny)
        hL, uL, vL, hR, uR, vR = (torch.where(mL, hR, hL), torch.where(mL, -uR, uL), torch.where(mL, -vR, vL),
                                  torch.where(mR, hL, hR), torch.where(mR, -uL, uR), torch.where(mR, -vL, vR))
        a, b = torch.sqrt(hL + EPS), torch.sqrt(hR + EPS)
        ur, vr = (a * uL / hL + b * uR / hR) / (a + b), (a * vL / hL + b * vR / hR) / (a + b)
        un = ur * nx + vr * ny
        c = torch.sqrt(G * 0.5 * (hL + hR) + EPS)
        e0, e1, e2 = xR - xL, uR - uL, vR - vL
        jump = (e1 * nx + e2 * ny - un * e0) / (2 * c)
        w0 = (vr * nx - ur * ny) * e0 + ny * e1 - nx * e2
        mag = lambda x: torch.sqrt(x * x + EPS)  # noqa: E731
        a0, a1, a2 = mag(un) * w0, mag(un - c) * (0.5 * e0 - jump), mag(un + c) * (0.5 * e0 + jump)
        r = (a1 + a2, ny * a0 + (ur - c * nx) * a1 + (ur + c * nx) * a2, -nx * a0 + (vr - c * ny) * a1 + (vr + c * ny) * a2)
        nL, nR = (uL * nx + vL * ny) / hL, (uR * nx + vR * ny) / hR
        pr = 0.5 * G * ((xL + EPS) ** 2 + 2 * xL * sL + (xR + EPS) ** 2 + 2 * xR * sR)
        both = (nL * hL + nR * hR, nL * uL + nR * uR + pr * nx, nL * vL + nR * vR + pr * ny)
        return [torch.where(dL & dR, 0.0, torch.where(one, k, 0.5 * (s - q))) for k, s, q in zip(alone, both, r)]

    def step(self, Q, dt, n, **over):
        E = Q + dt * self.rhs(Q, n, **over)
        dry = E[:, :1] < H_SMALL
        low = torch.zeros(1, 3, 1, dtype=E.dtype, device=E.device)
        low[0, 0] = H_SMALL
        return torch.where(dry, low, E)

    def host(self, Q):
        return Q.transpose(0, 1).reshape(-1).cpu().numpy()


def _closure(flow):
    """n = 0.01 + softplus(MLP(h, |u|, zb)), one weight set of 353 per field."""
    def n(Q, w):
        h = Q[:, 0] + flow.hs
        wet = h > H_SMALL
        h = torch.where(wet, h, H_SMALL)
        u, v = torch.where(wet, Q[:, 1], 0.0) / h, torch.where(wet, Q[:, 2], 0.0) / h
        F = torch.stack([h, torch.sqrt(u * u + v * v + EPS), flow.zb.expand_as(h)], 1)
        a = torch.tanh(w[:, :48].reshape(-1, 16, 3) @ F + w[:, 48:64, None])
        a = torch.tanh(w[:, 64:320].reshape(-1, 16, 16) @ a + w[:, 320:336, None])
        return 0.01 + torch.nn.functional.softplus((w[:, 336:352, None] * a).sum(1) + w[:, 352:], threshold=700.0)
    return n


def _network(flow):
    """The roughness network of NET: Dense, tanh, LayerNorm twice, then a bounded output."""
    (lo, hi), (h0, h1) = NET["output_bounds"], NET["h_bounds"]

    def n(Q, w):
        h = Q[:, 0] + flow.hs
        x = (2 * (torch.where(h > H_SMALL, h, H_SMALL) - h0) / (h1 - h0) - 1)[:, None]
        at = 0
        for k in (1, 3):
            W, b, g, s = torch.split(w[at:at + 3 * k + 9], [3 * k, 3, 3, 3])
            at += 3 * k + 9
            x = torch.tanh(W.reshape(k, 3).T @ x + b[:, None])
            x = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + float(np.float32(1e-5)))
            x = x * g[:, None] + s[:, None]
        return lo + (hi - lo) * torch.sigmoid((w[at:at + 3, None] * x).sum(1) + w[at + 3])
    return n


def _gradient(flow, dt, steps, cotangent, n_of, par):
    """The final state and the cotangents of Q0 and of every entry of `par`; n_of(Q, par) is the roughness."""
    step = lambda Q, p: flow.step(Q, dt, n_of(Q, p), S0=p.get("S0"), zb=p.get("zb"), Qin=p.get("Qin"))  # noqa: E731
    with torch.no_grad():
        traj = [flow.Q0]
        for _ in range(steps):
            traj.append(step(traj[-1], par))
    flat = [(k, i) for k, v in par.items() for i in range(len(v) if isinstance(v, tuple) else 1)]
    sums, lam = None, cotangent(traj[-1])
    for Q in reversed(traj[:-1]):
        Q = Q.detach().requires_grad_()
        p = {k: tuple(x.detach().requires_grad_() for x in v) if isinstance(v, tuple) else v.detach().requires_grad_()
             for k, v in par.items()}
        wrt = [p[k][i] if isinstance(p[k], tuple) else p[k] for k, i in flat]
        lam, *got = torch.autograd.grad(step(Q, p), [Q] + wrt, lam, allow_unused=True)
        got = [torch.zeros_like(w) if g is None else g for g, w in zip(got, wrt)]
        sums = got if sums is None else [a + b for a, b in zip(sums, got)]
    return traj[-1], lam, {(k, i): v for (k, i), v in zip(flat, sums)}


def _bed_cotangent(flow, sums, extra):
    zb = flow.zb.detach().requires_grad_()
    g, = torch.autograd.grad(flow.bed_slope(zb), zb, [sums["S0", 0], sums["S0", 1]])
    return g + sums["zb", 0] + extra


def _tsit5(flow, n_of, Q, t_end, frames, dt, abstol=1e-6, reltol=1e-3):
    """Tsitouras' 5(4) pair (Comput. Math. Appl. 62, 2011), first same as last, steps landing on the frames."""
    a = [[0.161], [-0.008480655492356989, 0.335480655492357],
         [2.897153057105493, -6.359448489975075, 4.3622954328695815],
         [5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525],
         [5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401, -0.028269050394068383],
         [0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081, 2.324710524099774]]
    e = [-0.00178001105222577714, -0.0008164344596567469, 0.007880878010261995, -0.1447110071732629,
         0.5823571654525552, -0.45808210592918697, 0.015151515151515152]
    f = lambda q: flow.rhs(q, n_of(q))  # noqa: E731
    k0, t, out, counts = f(Q), 0.0, [flow.host(Q)], [0, 0, 1]
    for s in range(1, frames + 1):
        stop = t_end * s / frames
        while t < stop:
            last = dt >= (stop - t) * (1 - 1e-12)
            h = stop - t if last else dt
            k = [k0]
            for row in a:
                new = Q + sum(h * w * v for w, v in zip(row, k))
                k.append(f(new))
            counts[2] += 6
            err = sum(h * w * v for w, v in zip(e, k)) / (abstol + reltol * torch.maximum(Q.abs(), new.abs()))
            err = math.sqrt(float((err * err).mean()))
            fac = 0.9 * err ** -0.2 if err > 0 else 10.0
            if err <= 1:
                t, Q, k0 = (stop if last else t + h), new, k[-1]
                counts[0] += 1
                if not last or h * min(10.0, max(0.2, fac)) < dt:
                    dt = h * min(10.0, max(0.2, fac))
            else:
                counts[1] += 1
                dt = h * max(0.2, fac)
        out.append(flow.host(Q))
    return np.stack(out), np.array(counts)


def exact(case, seed):
    d = _inputs(case, seed)
    c, path, dt, steps, K = d["case"], case["path"], d["dt"], d["steps"], case.get("fields", 1)
    flow = _Flow(c, K)
    t = lambda v: torch.as_tensor(v, dtype=torch.float64, device=flow.dev)  # noqa: E731
    if path == "rhs":
        return flow.host(flow.rhs(flow.Q0, flow.n0))
    if path in ("step", "batch"):
        Q = flow.Q0
        for _ in range(steps):
            Q = flow.step(Q, dt, flow.n0)
        return flow.host(Q)
    if path == "tsit5":
        w = d["law"]
        n_of = lambda Q: w["n_lower"] + (w["n_upper"] - w["n_lower"]) / (  # noqa: E731
            1 + torch.exp(w["k"] * (torch.clamp(Q[:, 0] + flow.hs, min=H_SMALL) - w["h_mid"])))
        return _tsit5(flow, n_of, flow.Q0, dt * steps, case["frames"], dt)
    zone = torch.as_tensor(c.zone, dtype=torch.int64, device=flow.dev) if c.zone is not None else None
    if path == "tangent":
        n, dn = t(c.zone_n)[zone][None], t(d["dn"])[zone][None]
        Q, T = flow.Q0, torch.zeros_like(flow.Q0)
        for _ in range(steps):
            with torch.autograd.forward_ad.dual_level():
                dual = [torch.autograd.forward_ad.make_dual(*v) for v in ((Q, T), (n, dn))]
                Q, T = torch.autograd.forward_ad.unpack_dual(flow.step(dual[0], dt, dual[1]))
        return flow.host(Q), flow.host(T)
    if path in ("inversion", "network"):
        target = t(d["target"]).reshape(3, 1, -1).transpose(0, 1)
        par = {"zone": t(c.zone_n), "Qin": flow.Qin} if path == "inversion" else {"w": t(d["weights"])}
        net = _network(flow)
        n_of = (lambda Q, p: p["zone"][zone][None]) if path == "inversion" else (lambda Q, p: net(Q, p["w"]))
        QN, lam, sums = _gradient(flow, dt, steps, lambda Q: (Q - target) / d["N"], n_of, par)
        return (flow.host(QN), flow.host(lam)) + tuple(v.reshape(-1).cpu().numpy() for v in sums.values())
    probe = torch.as_tensor(d["probe"][:len(d["probe"]) // K].astype(np.int64), device=flow.dev)
    target = t(d["target"]).reshape(K, -1)
    miss = lambda Q: (Q[:, 0] + flow.hs + flow.zb)[:, probe] - target  # noqa: E731

    def cotangent(Q):
        lam = torch.zeros_like(Q)
        lam[:, 0, probe] = 2 * miss(Q)
        return lam

    if path == "gradient":
        par = {"n": t(d["n"])[None], "zb": flow.zb, "S0": flow.S0, "Qin": flow.Qin}
        QN, lam, sums = _gradient(flow, dt, steps, cotangent, lambda Q, p: p["n"], par)
        got = {"n": lambda: sums["n", 0].reshape(-1),
               "zb": lambda: _bed_cotangent(flow, sums, cotangent(QN)[0, 0]),
               "Q": lambda: sums["Qin", 0].reshape(-1)}
        return [float((miss(QN) ** 2).sum())] + [got[k]().cpu().numpy() for k in ("n", "zb", "Q") if k in case["wrt"].split()]
    net = _closure(flow)
    QN, lam, sums = _gradient(flow, dt, steps, cotangent, lambda Q, p: net(Q, p["w"]), {"w": t(d["weights"]), "Qin": flow.Qin})
    return float((miss(QN) ** 2).sum()), sums["Qin", 0].reshape(-1).cpu().numpy(), sums["w", 0].reshape(-1, 353).squeeze().cpu().numpy()

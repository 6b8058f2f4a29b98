"""The work whose speed matters to a user of this framework, through its
public entry points.

Five kinds of call:

* ``solve``: one mesh in an ``Environment``: ``calls`` x ``env.step(steps)``,
  then the fields a program reads afterwards (``read``: the pdf; the moments
  and node fields for a plot; or every observable).
* ``batch``: ``BatchSolver`` on several porous channels, started from node
  fields (a warm start), run with per-case residual checks, read back.
* ``predict``: the shipped network's prediction for several porous cases,
  host inputs included (what a warm start pays before it solves).
* ``train``: one training step's forward and backward pass of the network
  over a batch of meshes; returns the loss and every gradient.
* ``layer``: one message-passing layer, aggregation and dense block, forward
  and backward, on one graph.

Meshes are fixed by a case's own values and built once per process, as a
program meshes once and solves many times; the fields, inlet speeds, node
features and targets follow the seed.
"""
from __future__ import annotations

import dataclasses
import functools
import importlib
import math
import os

import numpy as np
import torch
import torch.utils.checkpoint

fv = importlib.import_module("fvdbm-jax_amd")
batch_mod = importlib.import_module("fvdbm-jax_amd.batch")
surrogate = importlib.import_module("fvdbm-jax_amd.surrogate")
meshgen, porous = fv.meshgen, fv.porous

WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(fv.__file__)), "data", "surrogate_porous.npz")


def listed():
    return [
        # the documented idiom, one call per step, on the 32x32 cavity: call
        # and launch latency
        dict(name="cavity_stepwise", kind="solve", mesh="cavity", cells=2048, precision="fp32",
             scheme="upwind", lattice="d2q9", calls=100, steps=1, read="moments"),
        # the README's run of the cavity: 1000 steps in one call, then every field
        dict(name="cavity_1000", kind="solve", mesh="cavity", cells=2048, precision="fp32",
             scheme="upwind", lattice="d2q9", calls=1, steps=1000, read="all"),
        # an ordinary single porous channel (the middle of the 20k-200k range)
        dict(name="porous_60k", kind="solve", mesh="porous", cells=60_001, precision="fp32",
             scheme="upwind", lattice="d2q9", calls=1, steps=1000, read="moments"),
        # a cylinder channel at a quarter of the benchmark's size
        dict(name="channel_250k", kind="solve", mesh="channel", cells=250_000, precision="fp32",
             scheme="upwind", lattice="d2q9", calls=1, steps=1000, read="pdf"),
        # the benchmark's 1M-cell cylinder channel
        dict(name="channel_1m", kind="solve", mesh="channel", cells=1_000_000, precision="fp32",
             scheme="upwind", lattice="d2q9", calls=1, steps=2000, read="pdf"),
        # the double-precision twin that states the FP32 error
        dict(name="channel_fp64", kind="solve", mesh="channel", cells=150_000, precision="fp64",
             scheme="upwind", lattice="d2q9", calls=1, steps=400, read="pdf"),
        # the second-order flux, on the cavity (it is not stable on the channels'
        # scales), 201 x 201 squares
        dict(name="cavity_lw", kind="solve", mesh="cavity", cells=80_802, precision="fp32",
             scheme="lax_wendroff", lattice="d2q9", calls=1, steps=1000, read="pdf"),
        # the 13-velocity lattice
        dict(name="channel_d2q13", kind="solve", mesh="channel", cells=250_000, precision="fp32",
             scheme="upwind", lattice="d2q13", calls=1, steps=500, read="pdf"),
        # a batch of porous channels warm-started from node fields, checked
        # every 500 steps
        dict(name="batch_16", kind="batch", cases=16, low=20_000, high=90_000, first=0, steps=1000,
             check=500),
        # warm-start predictions for a group of cases
        dict(name="predict_12", kind="predict", cases=12, low=20_000, high=90_000, first=100),
        # a training step: 16 meshes, about 0.5M graph nodes
        dict(name="train_16", kind="train", cases=8, copies=2, low=20_000, high=110_000, first=200),
        # one layer on one mid-size graph of an odd node count
        dict(name="layer_45k", kind="layer", cells=90_001, first=300),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["solve"] * 6 + ["batch", "predict", "train", "layer", "layer"])
    first = rng.randrange(1000, 900_000)
    if kind == "batch":
        low = _log_int(rng, 6_000, 40_000)
        return dict(kind=kind, cases=rng.randint(2, 14), low=low, high=2 * low + 1, first=first,
                    steps=rng.randint(200, 900), check=rng.choice([100, 250, 333, 500]))
    if kind == "predict":
        low = _log_int(rng, 4_000, 40_000)
        return dict(kind=kind, cases=rng.randint(1, 10), low=low, high=2 * low + 1, first=first)
    if kind == "train":
        low = _log_int(rng, 4_000, 40_000)
        return dict(kind=kind, cases=rng.randint(1, 7), copies=rng.randint(1, 2), low=low,
                    high=2 * low + 1, first=first)
    if kind == "layer":
        return dict(kind=kind, cells=_log_int(rng, 3_000, 200_000), first=first)
    mesh = rng.choice(["cavity", "porous", "channel", "channel"])
    scheme = rng.choice(["upwind", "lax_wendroff"]) if mesh == "cavity" else "upwind"
    if mesh == "cavity":
        cells = 2 * _log_int(rng, 12, 240) ** 2
    elif mesh == "porous":
        cells = _log_int(rng, 8_000, 200_000)
    else:
        cells = _log_int(rng, 4_000, 600_000)
    lattice = rng.choice(["d2q9", "d2q9", "d2q9", "d2q13"])
    calls = rng.choice([1, 1, 1, 20])
    most = min(1000, 250_000_000 // cells)
    steps = rng.randint(1, 3) if calls > 1 else rng.randint(max(most // 4, 1), most)
    return dict(kind="solve", mesh=mesh, cells=cells, precision=rng.choice(["fp32", "fp32", "fp32", "fp64"]),
                scheme=scheme, lattice=lattice,
                calls=calls, steps=steps, read=rng.choice(["pdf", "moments", "all"]))


# ---------------------------------------------------------------------------
# meshes (fixed by the case, built once per process)
# ---------------------------------------------------------------------------
def _mesher(raw):
    m = fv.Mesher.from_raw(raw)
    m.enforce_ccw()
    m.calc_mesh_properties()
    return m


@functools.lru_cache(maxsize=None)
def _mesh(kind, cells):
    if kind == "cavity":
        return _mesher(meshgen.ldc_structured(int(round(math.sqrt(cells / 2)))))
    if kind == "porous":
        return _mesher(meshgen.porous_channel(7, target_cells=cells, n_obstacles=6, r_range=(0.02, 0.06),
                                              gap=0.03))
    return _mesher(meshgen.cylinder_channel(cells, seed=1))


@functools.lru_cache(maxsize=None)
def _porous_case(seed, cells):
    return porous.make_case(seed, porous.STEADY, target_cells=cells)


def _members(case):
    """(seed, target cells) of a group's porous cases: sizes spread evenly over [low, high], odd."""
    n, low, high = case["cases"], case["low"], case["high"]
    return [(case["first"] + i, (low + (high - low) * i // max(n - 1, 1)) | 1) for i in range(n)]


def _porous_group(case):
    return [_porous_case(*m) for m in _members(case)]


def _containers(case, seed):
    """Containers with boundary conditions and a start state, of one mesh: a
    cavity with a moving lid, or a channel with a parabolic inlet."""
    m = _mesh(case["mesh"], case["cells"])
    rng = np.random.default_rng(seed)
    lattice = fv.D2Q13 if case["lattice"] == "d2q13" else fv.D2Q9
    zero = np.array([0.0, 0.0])
    if case["mesh"] == "cavity":
        dyn = lattice(tau=0.6, delta_t=0.01)
        c, f, n = m.to_env(dyn, case["scheme"], dim_multiplier=1)
        n = m.set_vel_node(n, meshgen.LID, np.array([rng.uniform(0.05, 0.1), 0.0]))
        n = m.set_vel_node(n, meshgen.WALL, zero)
    else:
        tau = 0.55 if case["mesh"] == "channel" else 0.7
        height = 0.41 if case["mesh"] == "channel" else porous.HEIGHT
        scale = 1.0 if case["mesh"] == "channel" else porous.SCALE
        u_max = rng.uniform(0.05, 0.1) if case["mesh"] == "channel" else rng.uniform(0.02, 0.05)
        dyn = lattice(tau=tau, delta_t=1.0)
        c, f, n = m.to_env(dyn, case["scheme"], dim_multiplier=1.0 / (scale * porous.mean_area(m)))
        dt = porous.stable_dt(m, f.L, tau)
        dyn.delta_t = float(np.float32(dt / math.sqrt(2.0) if case["lattice"] == "d2q13" else dt))
        n = m.set_vel_profile(n, meshgen.INLET, lambda p: meshgen.parabolic_inlet(p[:, 1], height, u_max))
        n = m.set_rho_node(n, meshgen.OUTLET, 1.0)
        n = m.set_vel_node(n, meshgen.WALL, zero)
        n = m.set_vel_node(n, meshgen.OBSTACLE, zero)
    rho, vel = _smooth_fields(c.centers, rng)
    c.pdf = _equilibrium(dyn, rho, vel).astype(np.float64 if case["precision"] == "fp64" else np.float32)
    return c, f, n


def _smooth_fields(xy, rng):
    """rho near 1 and a speed of a few percent, a handful of waves over the domain."""
    rho = np.ones(len(xy))
    vel = np.zeros((len(xy), 2))
    for _ in range(4):
        kx, ky = rng.uniform(1.0, 12.0, 2)
        a, b, d = rng.uniform(0.0, 2 * np.pi, 3)
        s = kx * xy[:, 0] + ky * xy[:, 1]
        rho += 0.002 * np.sin(s + a)
        vel[:, 0] += 0.01 * np.sin(s + b)
        vel[:, 1] += 0.005 * np.sin(s + d)
    return rho, vel


def _equilibrium(dyn, rho, vel):
    """The quadratic equilibrium of the lattice, in 64 bits."""
    ksi = np.asarray(dyn.KSI, np.float64)
    c2 = float(dyn.C) ** 2
    cu = vel @ ksi.T
    uu = (vel * vel).sum(1, keepdims=True)
    return np.asarray(dyn.W, np.float64) * rho[:, None] * (1 + cu / c2 + cu * cu / (2 * c2 * c2) - uu / (2 * c2))


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_solve(case, seed):
    c, f, n = _containers(case, seed)
    env = fv.Environment(c, f, n, precision=case["precision"])
    env.init()
    return dict(kind="solve", env=env, calls=case["calls"], steps=case["steps"], read=case["read"])


def _run_solve(s):
    env = s["env"]
    for _ in range(s["calls"]):
        env = env.step(s["steps"])
    out = {"pdf": env.cells.pdf}
    if s["read"] in ("moments", "all"):
        out["rho"], out["vel"] = env.cells.rho, env.cells.vel
        out["node_rho"], out["node_vel"] = env.nodes.rho, env.nodes.vel
    if s["read"] == "all":
        out["pdf_eq"], out["flux"], out["node_pdf"] = env.cells.pdf_eq, env.faces.pdf, env.nodes.pdf
    return out


def _node_fields(group, seed):
    rng = np.random.default_rng(seed)
    fields = [_smooth_fields(c.mesher.points, rng) for c in group]
    return (np.concatenate([r for r, _ in fields]).astype(np.float32),
            np.concatenate([v for _, v in fields]).astype(np.float32))


def _prepare_batch(case, seed):
    group = _porous_group(case)
    rho, vel = _node_fields(group, seed)
    solver = batch_mod.BatchSolver([c.env_tuple() for c in group])
    return dict(kind="batch", solver=solver, rho=rho, vel=vel, steps=case["steps"], check=case["check"])


def _run_batch(s):
    b = s["solver"]
    b.init_equilibrium_nodes(s["rho"], s["vel"])
    b.set_active(np.ones(b.n, np.int32), reset_steps=True)
    st = b.run(s["steps"], s["check"], 1e-6, 100.0)
    rho, vel = b.node_fields()
    return {"rho": rho, "vel": vel, "pdf": b.get_pdf(), "residual": st["residual"], "steps": st["steps"]}


def _prepare_predict(case, seed):
    rng = np.random.default_rng(seed)
    group = [dataclasses.replace(c, u_in=float(rng.uniform(0.02, 0.05)),
                                 dynamics=fv.D2Q9(float(rng.uniform(0.55, 0.9)), c.dynamics.delta_t))
             for c in _porous_group(case)]
    return dict(kind="predict", net=surrogate.MeshNet.load(WEIGHTS), group=group)


def _run_predict(s):
    out = s["net"].predict(s["group"])
    return {"rho": [r for r, _ in out], "vel": [v for _, v in out]}


@functools.lru_cache(maxsize=None)
def _inputs(seed, cells):
    return surrogate.case_inputs(_porous_case(seed, cells), (32, 16), True)


def _prepare_train(case, seed):
    rng = np.random.default_rng(seed)
    samples = []
    for _ in range(case["copies"]):
        for member in _members(case):
            c = _porous_case(*member)
            x, g, n = _inputs(*member)
            x = x.copy()  # another inlet speed and tau, as another case on the same geometry
            x[:, 7] = rng.uniform(-1.6, 1.6)
            x[:, 8] = rng.uniform(-1.7, 1.7)
            rho, vel = _smooth_fields(c.mesher.points, rng)
            y = np.zeros((g["n"], 3), np.float32)
            y[:n, 0], y[:n, 1:] = 100 * (rho - 1), 30 * vel
            samples.append(surrogate.device_sample(x, g, y, n))
    return dict(kind="train", net=surrogate.MeshNet.load(WEIGHTS), samples=samples)


def _run_train(s):
    net = s["net"]
    x, g, y, m = surrogate.concat_device(s["samples"])
    for p in net.parameters():
        p.grad = None
    loss = torch.sum(m * (net(x, g) - y) ** 2) / (3.0 * torch.sum(m))
    loss.backward()
    return {"loss": loss.detach(), **{k: p.grad for k, p in net.params.items()}}


def _prepare_layer(case, seed):
    _, g, _ = _inputs(case["first"], case["cells"])
    gen = torch.Generator(device="cuda").manual_seed(seed)
    h = torch.randn((g["n"], 64), generator=gen, device="cuda")
    dy = torch.randn((g["n"], 64), generator=gen, device="cuda")
    weights = [w.detach().requires_grad_() for w in surrogate.MeshNet.load(WEIGHTS).block("proc2")]
    return dict(kind="layer", h=h.requires_grad_(), dy=dy, weights=weights, g=surrogate.graph_to_device(g))


def _run_layer(s):
    y = surrogate.mlp2(surrogate.aggregate(s["h"], s["g"]), *s["weights"])
    grads = torch.autograd.grad(y, [s["h"]] + s["weights"], s["dy"])
    return {"y": y.detach(), **dict(zip(("dh", "dw1", "db1", "dw2", "db2"), grads))}


_PREPARE = dict(solve=_prepare_solve, batch=_prepare_batch, predict=_prepare_predict,
                train=_prepare_train, layer=_prepare_layer)
_RUN = dict(solve=_run_solve, batch=_run_batch, predict=_run_predict, train=_run_train,
            layer=_run_layer)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# per cell: 1.5 faces (normal, length, two cells, two nodes), half a node
# (2 values and a list of 6 cells with distances)
def _mesh_bytes(cells, es):
    return cells * (1.5 * (3 * es + 16) + 0.5 * (2 * es + 6 * (4 + es)))


# operations of one cell update: 3 faces of Q - 1 products with the pdf, the
# length and the sum, the moments, the equilibrium (about 8 per velocity) and
# the relaxation (5 per velocity); Lax-Wendroff interpolates (5 more per term)
def _step_flops(q, scheme):
    return 3 * (q - 1) * (3 if scheme == "upwind" else 8) + 3 * q + 13 * q


def work(case):
    kind = case["kind"]
    if kind == "solve":
        es, q = (8 if case["precision"] == "fp64" else 4), (13 if case["lattice"] == "d2q13" else 9)
        c, n = case["cells"], case["calls"] * case["steps"]
        out = {"pdf": q, "moments": q + 3 + 1.5, "all": q + 3 + 1.5 + q + 1.5 * q + 0.5 * q}[case["read"]]
        return dict(bytes=c * es * (q + out) + _mesh_bytes(c, es), flops=c * n * _step_flops(q, case["scheme"]))
    if kind == "layer":
        n = case["cells"] / 2 + 700
        e = n * 8.2
        dense = 2 * (256 * 64 + 64 * 64)
        return dict(bytes=n * 64 * 4 * 4 + 2 * e * 16 + 2 * 4 * (256 * 64 + 64 * 64),
                    flops=n * 3 * dense + 2 * e * 64 * 6)
    cells = sum(size for _, size in _members(case))
    if kind == "batch":
        return dict(bytes=cells * 4 * (9 + 1.5 + 1.5) + _mesh_bytes(cells, 4),
                    flops=cells * case["steps"] * _step_flops(9, "upwind"))
    n = (cells / 2 + 600 * case["cases"]) * case.get("copies", 1)
    e = n * 8.2
    forward = n * 2 * (16 * 64 + 64 * 64 + 6 * (256 * 64 + 64 * 64) + 64 * 64 + 64 * 16) + 6 * e * 64 * 6
    if kind == "predict":
        return dict(bytes=n * 4 * (16 + 3) + e * 16, flops=forward)
    return dict(bytes=n * 4 * (16 + 3 + 1) + e * 28, flops=3 * forward)


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed) if case["kind"] in _EXACT else None


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Flow:
    """One mesh's step in 64 bits: moments and equilibrium, boundary-node
    pdfs by inverse-distance weighting, face fluxes with ghosts, cell update."""

    def __init__(self, c, f, n, precision):
        d = self.d = _device()
        wide = precision == "fp64"

        def real(a):
            return torch.as_tensor(np.asarray(a, np.float64), device=d)

        def index(a):
            return torch.as_tensor(np.asarray(a, np.int64), device=d)

        dyn = c.dynamics
        self.q = int(dyn.NUM_QUIVERS)
        self.ksi = real(dyn.KSI)
        if self.q == 9:
            w = [4 / 9] + [1 / 9] * 4 + [1 / 36] * 4
            self.c2 = 1.0 / 3.0
        else:
            w = [3 / 8] + [1 / 12] * 4 + [1 / 16] * 4 + [1 / 96] * 4
            self.c2 = 0.5
        self.w = real(w)
        self.tau, self.dt = float(dyn.tau), float(dyn.delta_t)
        self.upwind = f.flux_scheme == "upwind"
        self.cell_faces = index(c.face_indices)
        self.signs = real(c.face_normals)
        cells = index(f.stencil_cells_index)
        dist = real(f.stencil_dists_f64 if wide else f.stencil_dists)
        normal = real(f.n_f64 if wide else f.n)
        self.length = real(f.L_f64 if wide else f.L).reshape(-1, 1)
        self.phi = normal @ self.ksi.T
        nodes = index(f.nodes_index)
        ghost = (cells < 0).any(1)
        self.gf = torch.nonzero(ghost)[:, 0]
        gc = cells[self.gf]
        self.g_left = gc[:, 0] < 0
        self.known = torch.where(self.g_left, gc[:, 1], gc[:, 0])
        gd = dist[self.gf]
        self.ratio = torch.where(self.g_left, gd[:, 0] / gd[:, 1], gd[:, 1] / gd[:, 0])[:, None]
        self.gn = nodes[self.gf]
        self.a, self.b = cells[:, 0].clamp(min=0), cells[:, 1].clamp(min=0)
        s = dist.sum(1, keepdim=True)
        if not self.upwind:
            self.interp = dist[:, :1] / s - self.phi * self.dt / (2 * s)
        # slots of the state extended by the ghosts: each face value's source
        ghosts = torch.arange(len(self.gf), device=d) + len(self.cell_faces)
        left, right = self.a.clone(), self.b.clone()
        left[self.gf] = torch.where(self.g_left, ghosts, left[self.gf])
        right[self.gf] = torch.where(self.g_left, right[self.gf], ghosts)
        self.left, self.right = left, right
        if self.upwind:
            side = torch.where(self.phi >= 0, left[:, None], right[:, None])
            self.source = side * self.q + torch.arange(self.q, device=d)
        kind = torch.as_tensor(np.asarray(n.type).reshape(-1), device=d)
        nc = index(n.cells_index)
        nd = real(n.cell_dists_f64 if wide else n.cell_dists)
        weight = torch.where(nc >= 0, 1.0 / nd, torch.zeros_like(nd))
        self.active = []
        for t in (1, 2):
            at = torch.nonzero(kind == t)[:, 0]
            wt = weight[at]
            self.active.append((at, nc[at].clamp(min=0), (wt / wt.sum(1, keepdim=True))[:, :, None]))
        self.node_rho = real(n.rho_f64 if wide else n.rho).reshape(-1, 1).clone()
        self.node_vel = real(n.vel_f64 if wide else n.vel).reshape(-1, 2).clone()
        self.node_pdf = self.w.repeat(len(kind), 1)
        self.pdf = real(c.pdf)

    def equilibrium(self, rho, vel):
        c2 = self.c2
        cu = vel @ self.ksi.T
        uu = (vel * vel).sum(1, keepdim=True)
        s = 1 + cu / c2 + cu * cu / (2 * c2 * c2) - uu / (2 * c2)
        if self.q == 13:
            s = s + cu ** 3 / (2 * c2 ** 3) - 3 * cu * uu / (2 * c2 * c2)
        return self.w * rho * s

    def step(self):
        f = self.pdf
        self.rho = f.sum(1, keepdim=True)
        self.vel = (f @ self.ksi) / self.rho
        self.eq = self.equilibrium(self.rho, self.vel)
        for t, (at, nc, wt) in enumerate(self.active):
            if t == 0:
                self.node_rho[at] = (self.rho[nc] * wt).sum(1)
            else:
                self.node_vel[at] = (self.vel[nc] * wt).sum(1)
            self.node_pdf[at] = (self.equilibrium(self.node_rho[at], self.node_vel[at])
                                 + ((f[nc] - self.eq[nc]) * wt).sum(1))
        mean = 0.5 * (self.node_pdf[self.gn[:, 0]] + self.node_pdf[self.gn[:, 1]])
        full = torch.cat([f, mean + (mean - f[self.known]) * self.ratio])
        if self.upwind:
            value = full.reshape(-1)[self.source]
        else:
            value = full[self.left]
            value = value + (full[self.right] - value) * self.interp
        self.flux = value * self.phi * self.length
        total = sum(self.flux[self.cell_faces[:, k]] * self.signs[:, k:k + 1] for k in range(3))
        self.pdf = f + self.dt * ((self.eq - f) / self.tau - total)


def _exact_solve(case, seed):
    flow = _Flow(*_containers(case, seed), case["precision"])
    for _ in range(case["calls"] * case["steps"]):
        flow.step()
    out = {"pdf": flow.pdf}
    if case["read"] in ("moments", "all"):
        out["rho"], out["vel"] = flow.rho, flow.vel
        out["node_rho"], out["node_vel"] = flow.node_rho, flow.node_vel
    if case["read"] == "all":
        out["pdf_eq"], out["flux"], out["node_pdf"] = flow.eq, flow.flux, flow.node_pdf
    return out


def _exact_batch(case, seed):
    group = _porous_group(case)
    rho, vel = _node_fields(group, seed)
    out = {"rho": [], "vel": [], "pdf": [], "residual": []}
    o = 0
    for c in group:
        flow = _Flow(*c.env_tuple(), "fp32")
        d, n = flow.d, c.n_nodes
        nr = torch.as_tensor(rho[o:o + n], device=d).double()
        nv = torch.as_tensor(vel[o:o + n], device=d).double()
        o += n
        nc = torch.as_tensor(np.asarray(c.nodes.cells_index, np.int64), device=d)
        nd = torch.as_tensor(np.asarray(c.nodes.cell_dists, np.float64), device=d)
        w = torch.where(nc >= 0, 1.0 / nd, torch.zeros_like(nd))
        at = nc.clamp(min=0).reshape(-1)
        # node -> cell: the weights of a cell's vertices
        node = torch.cat([nr[:, None], nv, torch.ones_like(nr)[:, None]], 1)
        s = torch.zeros((c.n_cells, 4), dtype=torch.float64, device=d)
        s.index_add_(0, at, (node[:, None, :] * w[:, :, None]).reshape(-1, 4))
        s = s[:, :3] / s[:, 3:]
        flow.pdf = flow.equilibrium(s[:, :1], s[:, 1:])
        for _ in range(case["steps"]):
            flow.step()
        r2 = flow.pdf.sum(1, keepdim=True)
        v2 = (flow.pdf @ flow.ksi) / r2
        out["residual"].append(torch.linalg.norm(v2 - flow.vel) / torch.linalg.norm(v2))
        w = (w / w.sum(1, keepdim=True))[:, :, None]
        out["rho"].append((r2[nc.clamp(min=0)] * w).sum(1)[:, 0])
        out["vel"].append((v2[nc.clamp(min=0)] * w).sum(1))
        out["pdf"].append(flow.pdf)
    return {"rho": torch.cat(out["rho"]), "vel": torch.cat(out["vel"]), "pdf": torch.cat(out["pdf"]),
            "residual": torch.stack(out["residual"]), "steps": None}


def _dense(x, w1, b1, w2, b2):
    return torch.nn.functional.silu(x @ w1 + b1) @ w2 + b2


def _gather_means(h, g):
    off, col = g["off"].long(), g["col"].long()
    src = torch.repeat_interleave(torch.arange(len(off) - 1, device=h.device), off[1:] - off[:-1])
    hw = h[col] * g["w"].double()[:, None]
    parts = [h]
    for s in (None, g["ex"], g["ey"]):
        v = hw if s is None else hw * s.double()[:, None]
        parts.append(torch.zeros_like(h).index_add(0, src, v))
    return torch.cat(parts, 1)


def _exact_layer(case, seed):
    s = _prepare_layer(case, seed)
    h = s["h"].detach().double().requires_grad_()
    weights = [w.detach().double().requires_grad_() for w in s["weights"]]
    y = _dense(_gather_means(h, s["g"]), *weights)
    grads = torch.autograd.grad(y, [h] + weights, s["dy"].double())
    return {"y": y.detach(), **dict(zip(("dh", "dw1", "db1", "dw2", "db2"), grads))}


def _exact_train(case, seed):
    s = _prepare_train(case, seed)
    x, g, y, m = surrogate.concat_device(s["samples"])
    p = {k: v.detach().double().requires_grad_() for k, v in s["net"].params.items()}

    def block(name, v):
        return _dense(v, *(p[f"{name}.{k}"] for k in ("w1", "b1", "w2", "b2")))

    def layer(name, v):
        return v + block(name, _gather_means(v, g))

    h = block("enc", x.double())
    for k in range(s["net"].layers):
        h = torch.utils.checkpoint.checkpoint(layer, f"proc{k}", h, use_reentrant=False)
    loss = torch.sum(m.double() * (block("dec", h)[:, :3] - y.double()) ** 2) / (3.0 * torch.sum(m.double()))
    loss.backward()
    return {"loss": loss.detach(), **{k: v.grad for k, v in p.items()}}


_EXACT = dict(solve=_exact_solve, batch=_exact_batch, layer=_exact_layer, train=_exact_train)

"""What a user of this library has it do, as cases that can be timed.

Every case goes through the public entry points of ``molla_amd.MpmSimulation``:

* ``frame``     one frame of a running scene: ``step_n`` (or its graph replay),
                then positions, velocities and deformation into HBM buffers;
* ``wheel``     one control step of a driven wheel in soil: a new pose, a few
                substeps, the wrench and the positions back on the host;
* ``rollouts``  one round of data generation: a batch of scenes set from host
                arrays, stepped, and read back;
* ``identify``  one iteration of system identification: state and Young's
                moduli set, forward with checkpoints, loss gradient in HBM,
                reverse pass;
* ``keys``      the tile keys and the stable order of a particle set.

Scenes come from ``molla_amd.workloads`` or are boxes of soil, snow or an
elastic solid in the ``MpmConfig`` presets.  ``exact`` is the same physics in
64-bit torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from molla_amd import MpmSimulation, workloads
from molla_amd.config import Explicit, Fluid, Implicit, MpmConfig, Sand, Snow, Viscous
from molla_amd.rigid import MpmPrescribedSolid, SolidCylinder

def listed():
    return [
        # a robot's wheel in a sandbox: the smallest call, every control step
        # waits for its wrench
        {"name": "wheel_control", "kind": "wheel", "particles": 6001, "grid": 32, "substeps": 4},
        # the reference's smallest scene: an interactive frame, launch-bound
        {"name": "cube_frame", "kind": "frame", "material": "elastic", "particles": 8192, "grid": 32,
         "substeps": 20, "dt": 1e-4},
        # bit-repeatable soil (the reference's fixed summation order), as used
        # between checkpoints and for regression runs
        {"name": "sand_repeatable", "kind": "frame", "material": "sand", "particles": 16384, "grid": 32,
         "substeps": 4, "dt": 1e-4, "mode": "deterministic"},
        # the calibrated sand preset: semi-implicit grid solve, 48^3
        {"name": "sand_implicit", "kind": "frame", "material": "sand_calibrated", "particles": 32768, "grid": 48,
         "substeps": 8, "dt": 5e-4, "jacobi": 3},
        # an ordinary production scene with a ragged grid and count: snow over
        # a viscous layer
        {"name": "snow_mixed", "kind": "frame", "material": "mixed", "particles": 200003, "grid": 61,
         "substeps": 16, "dt": 1e-4},
        # a soil bed in a large domain: the pool of active tiles
        {"name": "terrain_sparse", "kind": "frame", "material": "sand", "particles": 150001, "grid": 512,
         "substeps": 8, "dt": 1e-4, "tiles": 16384},
        # data generation: scenes of 1e3 to 6.4e4 particles set, stepped, read
        {"name": "rollouts_48", "kind": "rollouts", "scenes": 48, "substeps": 100},
        # the large scene: a fluid pool and elastic blocks, 2 M particles
        {"name": "large_scene", "kind": "frame", "material": "large", "particles": 2000000, "grid": 256,
         "substeps": 20, "dt": 5e-5},
        # 512 uneven scenes in one launch per substep, replayed from a graph
        {"name": "batch_512", "kind": "batch", "scenes": 512, "substeps": 16, "sort_every": 64},
        # gradient of one scene: 64 substeps, checkpoint every 16
        {"name": "identify_scene", "kind": "identify", "scenes": 1, "particles": 65536, "grid": 64,
         "substeps": 64, "every": 16},
        # gradients of a batch of scenes
        {"name": "identify_128", "kind": "identify", "scenes": 128, "particles": 0, "grid": 0, "substeps": 32,
         "every": 16},
        # keys and order of a large particle set for a caller's own passes
        {"name": "keys_2m", "kind": "keys", "particles": 2000000, "grid": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fitting_grid(rng, n, ppc=8.0):
    side = (n / ppc) ** (1.0 / 3.0)
    return int(math.ceil(max(20.0, 1.6 * side + 12.0))) + rng.randrange(0, 14)


def draw(rng):
    kind = rng.choice(["wheel", "frame", "frame", "repeatable", "implicit", "sparse", "rollouts", "large", "batch",
                       "identify", "identify_batch", "keys"])
    if kind == "wheel":
        return {"kind": "wheel", "particles": _log_int(rng, 1000, 24000), "grid": 32, "substeps": rng.randrange(1, 9)}
    if kind == "frame":
        n = _log_int(rng, 1000, 1000000)
        return {"kind": "frame", "material": rng.choice(["elastic", "sand", "snow", "mixed"]), "particles": n,
                "grid": _fitting_grid(rng, n), "substeps": rng.randrange(4, 21), "dt": 1e-4}
    if kind == "repeatable":
        n = _log_int(rng, 1000, 60000)
        return {"kind": "frame", "material": rng.choice(["elastic", "sand"]), "particles": n,
                "grid": _fitting_grid(rng, n), "substeps": rng.randrange(2, 6), "dt": 1e-4, "mode": "deterministic"}
    if kind == "implicit":
        n = _log_int(rng, 2000, 300000)
        return {"kind": "frame", "material": "sand_calibrated", "particles": n, "grid": _fitting_grid(rng, n),
                "substeps": rng.randrange(3, 12), "dt": 5e-4, "jacobi": rng.randrange(1, 6)}
    if kind == "sparse":
        return {"kind": "frame", "material": "sand", "particles": _log_int(rng, 4000, 400000),
                "grid": _log_int(rng, 128, 640), "substeps": rng.randrange(3, 12), "dt": 1e-4, "tiles": 32768}
    if kind == "rollouts":
        return {"kind": "rollouts", "scenes": rng.randrange(2, 48), "substeps": rng.randrange(20, 101)}
    if kind == "large":
        return {"kind": "frame", "material": "large", "particles": _log_int(rng, 500000, 3000000), "grid": 256,
                "substeps": rng.randrange(4, 21), "dt": 5e-5}
    if kind == "batch":
        return {"kind": "batch", "scenes": rng.randrange(8, 400), "substeps": rng.randrange(4, 17),
                "sort_every": rng.choice([16, 32, 64])}
    if kind == "identify":
        n = _log_int(rng, 3000, 120000)
        return {"kind": "identify", "scenes": 1, "particles": n, "grid": 64, "substeps": rng.randrange(8, 65),
                "every": rng.choice([8, 16])}
    if kind == "identify_batch":
        return {"kind": "identify", "scenes": rng.randrange(2, 100), "particles": 0, "grid": 0,
                "substeps": rng.randrange(8, 33), "every": rng.choice([8, 16])}
    return {"kind": "keys", "particles": _log_int(rng, 5000, 2000000), "grid": rng.choice([64, 96, 128, 250, 256])}


# ---------------------------------------------------------------- scenes
def _spin(x, centre, omega, stretch, fall):
    """A moving, deforming body: a fall, a rotation and a stretch about its centre."""
    r = x - centre
    v = np.cross(np.asarray(omega, np.float64), r) + np.asarray(stretch, np.float64) * r
    v[:, 1] -= fall
    return v.astype(np.float32)


def _box(case, rng):
    """A box of one of the preset materials: (config, x, v, material ids or None)."""
    n, G = case["particles"], case["grid"]
    kind = case["material"]
    ppc = 8.0
    base = {"elastic": MpmConfig.viscous().copy(youngs=1e4, poisson=0.2, rheology=Viscous(0.0, 0.0),
                                                boundary_friction=0.0),
            "sand": MpmConfig.sand(), "sand_calibrated": MpmConfig.sand_calibrated(), "snow": MpmConfig.snow(),
            "mixed": MpmConfig.snow()}[kind]
    dx = 0.05
    rho = {"elastic": 1000.0, "snow": 400.0, "mixed": 400.0}.get(kind, 1600.0)
    cells = n / ppc
    if case.get("tiles"):  # a bed four to six cells deep on the floor
        deep = 6.0 if n > 20000 else 4.0
        size = np.array([math.sqrt(cells / deep), deep, math.sqrt(cells / deep)])
        fall, low = 0.05, 3.2
    else:
        side = cells ** (1.0 / 3.0)
        size = np.array([side, side, side])
        fall, low = 0.5, 4.0
    limit = G - 8.0
    if size[0] > limit:  # a taller box where the ground plan is full
        size = np.array([limit, cells / limit ** 2, limit])
    lo = np.array([(G - size[0]) / 2, low, (G - size[2]) / 2])
    origin = (-0.5 * G * dx, 0.0, -0.5 * G * dx)
    x = (np.asarray(origin) + dx * (lo + size * rng.random((n, 3)))).astype(np.float32)
    centre = np.asarray(origin) + dx * (lo + size / 2)
    v = _spin(x.astype(np.float64), centre, (0.6, 1.1, -0.8), (0.5, -0.9, 0.35), fall)
    vol = dx ** 3 / ppc
    materials, mat = [], None
    if kind == "mixed":
        materials = [Snow(), Viscous(4.0, 8.0)]
        mat = (x[:, 1] < centre[1]).astype(np.uint32)
    step = Implicit(case["jacobi"]) if case.get("jacobi") else Explicit()
    cfg = base.copy(grid_size=G, cell_size=dx, grid_origin=origin, particle_mass=rho * vol, particle_volume=vol,
                    max_particles=n, time_step=step, materials=materials)
    return cfg, x, v, mat


def _wheel_scene(case, rng):
    """A sandbox (the sparse-grid tests' spacing) and a wheel half sunk in it."""
    n = case["particles"]
    G, dx = case["grid"], 0.0625
    vol = dx ** 3 / 8.0
    cfg = MpmConfig.sand().copy(grid_size=G, grid_origin=(-1.0, -1.0, -1.0), cell_size=dx, max_particles=n,
                                max_rigid=2, youngs=2.0e4, particle_volume=vol, particle_mass=vol * 1600.0)
    side = 14.0
    size = np.array([side, n / 8.0 / side ** 2, side])
    if size[1] > 22.0:
        size = np.array([math.sqrt(n / 8.0 / 16.0), 16.0, math.sqrt(n / 8.0 / 16.0)])
    lo = np.array([(G - size[0]) / 2, 3.1, (G - size[2]) / 2])
    x = (-1.0 + dx * (lo + size * rng.random((n, 3)))).astype(np.float32)
    v = _spin(x.astype(np.float64), np.array([0.0, -0.5, 0.0]), (0.2, 0.5, -0.3), (0.2, -0.4, 0.15), 0.05)
    top = -1.0 + dx * (lo[1] + size[1])
    wheel = MpmPrescribedSolid(SolidCylinder(0.22, 0.10), center=(0.02, float(top), -0.013),
                               orientation=(math.sqrt(0.5), 0.0, 0.0, math.sqrt(0.5)),
                               linear_velocity=(0.4, -0.2, 0.0), angular_velocity=(0.0, 0.0, -2.0))
    return cfg, x, v, wheel


def _redrawn(xs, rng):
    """Other particles in the same blocks."""
    return [(x.min(axis=0) + np.ptp(x, axis=0) * rng.random(x.shape)).astype(np.float32) for x in xs]


def _batch_scenes(case, seed):
    """(configs, x, v, dt) of the batched workload: its scenes, with particles and motion from the seed."""
    cfgs, xs, meta = workloads.batched_scenes(case["scenes"])
    rng = np.random.default_rng([seed, 12])
    xs = _redrawn(xs, rng)
    fall = rng.uniform(0.3, 0.7)
    vs = [_spin(x.astype(np.float64), x.mean(axis=0), (0.6, 1.1, -0.8), (0.5, -0.9, 0.35), fall) for x in xs]
    return cfgs, xs, vs, meta["dt"]


def _identify_scenes(case, seed):
    """(configs, x, v, E, F, dt): dropped blocks with a strained start, moduli by particle or by scene."""
    rng = np.random.default_rng([seed, 77])
    if case["scenes"] == 1:
        cfg, d, meta = workloads.diff_scene(case["particles"], seed=seed, grid=case["grid"])
        cfgs, xs, vs, E = [cfg], [d["x"]], [d["v"]], d["E"]
    else:
        cfgs, d, meta = workloads.batched_diff_scenes(case["scenes"])
        xs, vs = _redrawn(d["x"], rng), d["v"]
        E = np.concatenate([np.full(len(x), e * math.exp(rng.uniform(-0.1, 0.1)), np.float32)
                            for x, e in zip(xs, meta["e0"])])
    F = []
    for x in xs:
        # a smooth strain with three distinct stretches that vary over the block
        r = (x - x.mean(axis=0)) / (np.ptp(x, axis=0) + 1e-6)
        f = np.zeros((len(x), 3, 3))
        f[:, 0, 0], f[:, 1, 1], f[:, 2, 2] = 1.03 + 0.02 * r[:, 1], 0.95 + 0.02 * r[:, 0], 0.99 + 0.01 * r[:, 2]
        f += 0.02 * rng.standard_normal((3, 3)) * np.array([[0, 1, 1], [1, 0, 1], [1, 1, 0]])
        F.append(f)
    return cfgs, xs, vs, E, np.concatenate(F).astype(np.float32), meta["dt"]


def _target(x):
    """Observed final positions: the start moved by a small shear."""
    t = x.copy()
    t[:, 0] += 0.01 * x[:, 1]
    t[:, 1] -= 0.03
    t[:, 2] += 0.004
    return t


# ---------------------------------------------------------------- state
def _device():
    return torch.device("cuda")


def _fields(n, names):
    wide = {"position": 3, "velocity": 3, "F": 9}
    return {k: torch.empty((n, wide[k]), dtype=torch.float32, device=_device()) for k in names}


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 11])
    if kind == "frame":
        if case["material"] == "large":
            cfg, d, _ = workloads.large_scene(case["particles"], seed=seed, grid=case["grid"])
            sim = MpmSimulation(cfg)
            sim.set_particles(d["x"], d["v"])
            for k in ("mass", "volume", "material"):
                sim.write_field(k, d[k])
        else:
            cfg, x, v, mat = _box(case, rng)
            sim = MpmSimulation(cfg, tile_capacity=case["tiles"] if case.get("tiles") else None)
            sim.set_particles(x, v)
            if mat is not None:
                sim.set_particle_materials(mat)
        if case.get("mode"):
            sim.set_p2g_mode(case["mode"])
        return {"case": case, "sim": sim, "out": _fields(sim.n, ("position", "velocity", "F"))}
    if kind == "wheel":
        cfg, x, v, wheel = _wheel_scene(case, rng)
        sim = MpmSimulation(cfg)
        sim.set_particles(x, v)
        return {"case": case, "sim": sim, "wheel": wheel}
    if kind in ("batch", "rollouts"):
        cfgs, xs, vs, dt = _batch_scenes(case, seed)
        sim = MpmSimulation(cfgs)
        state = {"case": case, "sim": sim, "dt": dt}
        if kind == "rollouts":
            return {**state, "x": xs, "v": vs}
        sim.set_particles_batch(xs, vs)
        sim.set_sort_interval(case["sort_every"])
        return {**state, "out": _fields(sim.n, ("position", "velocity"))}
    if kind == "identify":
        cfgs, xs, vs, E, F, dt = _identify_scenes(case, seed)
        sim = MpmSimulation(cfgs)
        x = np.concatenate(xs)
        target = torch.from_numpy(_target(x)).to(_device())
        n = len(x)
        out = {"x": torch.empty((n, 3), device=_device()), "gx": torch.empty((n, 3), device=_device()),
               "gv": torch.empty((n, 3), device=_device()), "gE": torch.empty(n, device=_device()),
               "gml": torch.empty(2, dtype=torch.float64, device=_device())}
        return {"case": case, "sim": sim, "xs": xs, "vs": vs, "E": E, "F": F, "dt": dt, "target": target, "out": out}
    if kind == "keys":
        cfg, d, _ = workloads.large_scene(case["particles"], seed=seed, grid=case["grid"])
        if case["grid"] != 256:  # the scene's cells are placed for 256^3: the same particles over another grid
            cfg = cfg.copy(grid_size=case["grid"], cell_size=1.0 / case["grid"])
        sim = MpmSimulation(cfg)
        sim.set_particles(d["x"], d["v"])
        out = {k: torch.empty(sim.n, dtype=torch.int32, device=_device()) for k in ("keys", "ids")}
        return {"case": case, "sim": sim, "out": out}
    raise ValueError(kind)


def run(state):
    case, sim = state["case"], state["sim"]
    kind = case["kind"]
    if kind == "frame":
        sim.step_n(case["dt"], case["substeps"])
        for k, t in state["out"].items():
            sim.read_field_device(k, t.data_ptr())
        return state["out"]
    if kind == "batch":
        sim.step_n_graph(state["dt"], case["substeps"])
        for k, t in state["out"].items():
            sim.read_field_device(k, t.data_ptr())
        return state["out"]
    if kind == "wheel":
        sim.set_prescribed_solids([state["wheel"]])
        sim.step_n(1e-4, case["substeps"])
        wrench = np.array([f + t for f, t in sim.read_rigid_wrenches()], np.float32)
        return {"wrench": wrench, "position": sim.read_positions(), "velocity": sim.read_velocities()}
    if kind == "rollouts":
        sim.set_particles_batch(state["x"], state["v"])
        sim.step_n(state["dt"], case["substeps"])
        return {"position": sim.read_positions(), "velocity": sim.read_velocities()}
    if kind == "identify":
        out = state["out"]
        if case["scenes"] == 1:
            sim.set_particles(state["xs"][0], state["vs"][0])
        else:
            sim.set_particles_batch(state["xs"], state["vs"])
        sim.write_field("youngs", state["E"])
        sim.write_field("F", state["F"])
        sim.diff_forward(state["dt"], case["substeps"], case["every"])
        sim.read_field_device("position", out["x"].data_ptr())
        sim.synchronize()
        loss_gradient = (out["x"] - state["target"])
        torch.cuda.synchronize()
        sim.diff_backward_device(loss_gradient.data_ptr(), 0, out["gx"].data_ptr(), out["gv"].data_ptr(),
                                 out["gE"].data_ptr(), out["gml"].data_ptr())
        sim.synchronize()
        return out
    if kind == "keys":
        out = state["out"]
        sim.sort_keys_noalloc(out["keys"].data_ptr(), out["ids"].data_ptr(), sim.n)
        sim.synchronize()  # the call's scratch is shared by every handle of the device
        return out
    raise ValueError(kind)


def work(case):
    """Bytes: state (x, v, C, F: 24 words) read and written once per substep, as
    the benchmark's roofline counts it, and what goes in and out.  Flops: 1,545
    per particle-substep of the forward, from the large scene's counters, and
    about three times that for a reverse substep."""
    kind = case["kind"]
    if kind in ("batch", "rollouts"):
        n = int(case["scenes"] * (6.4e4 - 1e3) / math.log(64.0))  # mean of the log-uniform counts
    elif kind == "identify" and case["scenes"] > 1:
        n = int(case["scenes"] * (3.2e4 - 4e3) / math.log(8.0))
    else:
        n = case["particles"]
    if kind == "keys":
        return {"bytes": 20 * n, "flops": 12 * n}
    steps = case["substeps"]
    if kind == "identify":
        return {"bytes": n * (steps * (192 + 296) + 28 * 4 + 14 * 4), "flops": n * steps * 1545 * 4}
    moved = {"frame": 60, "batch": 24, "wheel": 24, "rollouts": 48}[kind]
    return {"bytes": n * (192 * steps + moved), "flops": n * steps * 1545}


# ---------------------------------------------------------------- 64-bit reference
class _Scenes:
    """Per-particle scene constants in 64 bits and the cells of all scenes in one array."""

    def __init__(self, cfgs, counts):
        dev = _device()
        f64 = lambda v: torch.tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        counts_t = torch.tensor(counts, device=dev)
        self.sid = torch.repeat_interleave(torch.arange(len(cfgs), device=dev), counts_t)
        G = [int(c.grid_size) for c in cfgs]
        self.G = torch.tensor(G, device=dev)
        self.base = torch.tensor(np.concatenate([[0], np.cumsum([g ** 3 for g in G])[:-1]]), device=dev)
        self.cells = int(sum(g ** 3 for g in G))
        self.origin = f64([[f32(o) for o in c.grid_origin] for c in cfgs])
        self.dx = f64([f32(c.cell_size) for c in cfgs])
        self.gravity = f64([f32(c.gravity_y) for c in cfgs])
        self.bf = f64([f32(c.boundary_friction) for c in cfgs])
        self.E = f64([f32(c.youngs) for c in cfgs])
        self.nu = f64([f32(c.poisson) for c in cfgs])
        self.floor_y = f64([f32(c.floor_y) for c in cfgs])
        self.floor_friction = f64([f32(c.floor_friction) for c in cfgs])
        per = lambda t: t[self.sid]  # noqa: E731
        self.p_origin, self.p_dx, self.p_G, self.p_base = per(self.origin), per(self.dx), per(self.G), per(self.base)
        self.offs = torch.tensor([[i, j, k] for k in range(3) for j in range(3) for i in range(3)], device=dev)

    def stencil(self, x):
        """Cell of each of the 27 nodes, its weight, its offset from the particle."""
        xp = (x - self.p_origin) / self.p_dx[:, None]
        b = torch.floor(xp.detach() - 0.5)
        fx = xp - b
        w = torch.stack([0.5 * (1.5 - fx) ** 2, 0.75 - (fx - 1.0) ** 2, 0.5 * (fx - 0.5) ** 2], -1)  # (n, axis, node)
        o = self.offs
        W = w[:, 0][:, o[:, 0]] * w[:, 1][:, o[:, 1]] * w[:, 2][:, o[:, 2]]
        d = (o.to(torch.float64) - fx[:, None]) * self.p_dx[:, None, None]
        c = b.long()[:, None] + o
        g = self.p_G[:, None]
        return self.p_base[:, None] + c[..., 0] + g * (c[..., 1] + g * c[..., 2]), W, d

    def p2g(self, cell, W, d, m, v, A):
        mom = m[:, None, None] * v[:, None] + sum(A[:, None, :, j] * d[..., j, None] for j in range(3))
        q = torch.cat([(W * m[:, None])[..., None], W[..., None] * mom], -1).reshape(-1, 4)
        grid = torch.zeros((self.cells, 4), dtype=torch.float64, device=q.device)
        return grid.index_add_(0, cell.reshape(-1), q)

    def g2p(self, gv, cell, W, d):
        g = gv[cell.reshape(-1)].reshape(*cell.shape, 3)
        wg = W[..., None] * g
        C = torch.stack([(wg * d[..., j, None]).sum(1) for j in range(3)], -1) * (4.0 / self.p_dx ** 2)[:, None, None]
        return wg.sum(1), C

    def where(self, idx):
        """Scene and coordinates of cells."""
        s = torch.searchsorted(self.base, idx, right=True) - 1
        r, g = idx - self.base[s], self.G[s]
        return s, r % g, (r // g) % g, r // (g * g)


def _mm(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _svd(F):
    """F = U diag(s) V^T for det F > 0, by cyclic Jacobi on F^T F."""
    A = _mm(F.transpose(1, 2), F)
    V = torch.eye(3, dtype=F.dtype, device=F.device).expand_as(F).clone()
    for _ in range(7):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            apq = A[:, p, q]
            live = apq.abs() > 1e-300
            th = torch.where(live, (A[:, q, q] - A[:, p, p]) / torch.where(live, 2 * apq, torch.ones_like(apq)),
                             torch.zeros_like(apq))
            sign = torch.where(th >= 0, 1.0, -1.0).to(F.dtype)
            t = torch.where(live, sign / (th.abs() + torch.sqrt(1 + th * th)), torch.zeros_like(th))
            c = 1 / torch.sqrt(1 + t * t)
            s = t * c
            for M in (A, V):
                mp, mq = M[:, :, p].clone(), M[:, :, q].clone()
                M[:, :, p], M[:, :, q] = c[:, None] * mp - s[:, None] * mq, s[:, None] * mp + c[:, None] * mq
            ap, aq = A[:, p].clone(), A[:, q].clone()
            A[:, p], A[:, q] = c[:, None] * ap - s[:, None] * aq, s[:, None] * ap + c[:, None] * aq
    s = torch.sqrt(torch.diagonal(A, dim1=1, dim2=2).clamp_min(1e-300))
    return _mm(F, V) / s[:, None], s, V


def _shader_run(cfgs, counts, x, v, dt, substeps, mass=None, vol=None, mat=None, body=None):
    """`substeps` substeps of the shader model; returns x, v, F and the last substep's wrench."""
    dev = _device()
    f32 = lambda a: torch.as_tensor(np.asarray(a, np.float32)).to(dev).to(torch.float64)  # noqa: E731
    sc = _Scenes(cfgs, counts)
    n = len(x)
    x, v = f32(x), f32(v)
    m = f32(mass) if mass is not None else f32([c.particle_mass for c in cfgs])[sc.sid]
    vol = f32(vol) if vol is not None else f32([c.particle_volume for c in cfgs])[sc.sid]
    dt = float(np.float32(dt))
    if mat is None:
        rows = f32([c.material_rows()[0] for c in cfgs])[sc.sid]
    else:
        rows = f32(cfgs[0].material_rows())[torch.as_tensor(np.asarray(mat, np.int64)).to(dev)]
    rheo = rows[:, 0].round()
    sand, snow, viscous, fluid = rheo == 0, rheo == 1, rheo == 2, rheo == 3
    some = {k: bool(t.any()) for k, t in (("sand", sand), ("snow", snow), ("solid", ~fluid))}
    E, nu = sc.E[sc.sid], sc.nu[sc.sid]
    mu, lam = E / (2 * (1 + nu)), E * nu / ((1 + nu) * (1 - 2 * nu))
    I3 = torch.eye(3, dtype=torch.float64, device=dev)
    C = torch.zeros((n, 3, 3), dtype=torch.float64, device=dev)
    F = I3.expand(n, 3, 3).clone()
    U, s = F.clone(), torch.ones((n, 3), dtype=torch.float64, device=dev)
    jp = torch.zeros(n, dtype=torch.float64, device=dev)
    iters = int(getattr(cfgs[0].time_step, "jacobi_iters", 0) or 0)
    wrench = None
    for _ in range(substeps):
        h = torch.where(snow, torch.exp((-rows[:, 4] * jp).clamp(-3, 3)),
                        torch.where(sand, torch.exp(jp.clamp(-3, 3)), torch.ones_like(jp)))
        mh, lh = torch.where(fluid, torch.zeros_like(mu), mu * h), torch.where(fluid, rows[:, 7], lam * h)
        sh = s.clamp(0.1, 10.0)
        J = sh.prod(1)
        tau = 2 * mh[:, None] * (sh - 1) * sh + (lh * (J - 1) * J)[:, None]
        A = m[:, None, None] * C - (dt * vol * 4 / sc.p_dx ** 2)[:, None, None] * _mm(U * tau[:, None], U.transpose(1, 2))
        cell, W, d = sc.stencil(x)
        grid = sc.p2g(cell, W, d, m, v, A)
        act = torch.nonzero(grid[:, 0] > 0)[:, 0]
        q = grid[act]
        del grid
        si, ix, iy, iz = sc.where(act)
        stuck = torch.zeros(len(act), dtype=torch.bool, device=dev)
        gv = torch.where((q[:, 0] > 1e-9)[:, None], q[:, 1:] / q[:, :1], torch.zeros_like(q[:, 1:]))
        live = q[:, 0] > 1e-9
        gv[:, 1] += torch.where(live, dt * sc.gravity[si], torch.zeros_like(gv[:, 1]))
        G = sc.G[si]
        for a, c in enumerate((ix, iy, iz)):
            for near, bound in ((c < 2, torch.clamp_min), (c >= G - 2, torch.clamp_max)):
                for b in range(3):
                    wall = bound(gv[:, a], 0.0) if b == a else gv[:, b] * sc.bf[si]
                    gv[:, b] = torch.where(near, wall, gv[:, b])
        if body is not None:
            node = sc.origin[si] + torch.stack([ix, iy, iz], 1) * sc.dx[si][:, None]
            arm = node - f32(body.center)
            qx, qy, qz, qw = [float(np.float32(t)) for t in body.orientation]
            nq = math.sqrt(qx * qx + qy * qy + qz * qz + qw * qw)
            inv = torch.tensor([-qx / nq, -qy / nq, -qz / nq], dtype=torch.float64, device=dev).expand_as(arm)
            t = 2 * torch.linalg.cross(inv, arm)
            local = arm + (qw / nq) * t + torch.linalg.cross(inv, t)
            stuck = (torch.hypot(local[:, 0], local[:, 2]) < float(np.float32(body.shape.radius))) & \
                (local[:, 1].abs() < float(np.float32(body.shape.half_width))) & live
            bv = f32(body.linear_velocity) + torch.linalg.cross(f32(body.angular_velocity).expand_as(arm), arm)
            imp = q[:, :1] * bv - q[:, 1:]
            imp[:, 1] -= q[:, 0] * sc.gravity[si] * dt
            force = torch.where(stuck[:, None], -imp / dt, torch.zeros_like(imp))
            wrench = torch.cat([force.sum(0), torch.linalg.cross(arm, force).sum(0)])[None]
            gv = torch.where(stuck[:, None], bv, gv)
        full = torch.zeros((sc.cells, 3), dtype=torch.float64, device=dev)
        full[act] = gv
        if iters:
            mass_at = torch.zeros(sc.cells, dtype=torch.float64, device=dev)
            mass_at[act] = q[:, 0]
            near = []
            for a, c in enumerate((ix, iy, iz)):
                stride = G ** a
                for step in (1, -1):
                    inside = (c + step >= 0) & (c + step < G)
                    j = torch.where(inside, act + step * stride, act)
                    near.append((j, inside & (mass_at[j] > 1e-9)))
            cnt = sum(ok.to(torch.float64) for _, ok in near)
            al = dt * dt * q[:, 0] * (sc.E[si] / 1500.0) / sc.dx[si] ** 2
            for _it in range(iters):
                me = full[act]
                avg = sum(torch.where(ok[:, None], full[j], torch.zeros_like(me)) for j, ok in near)
                avg = torch.where((cnt > 0)[:, None], avg / cnt.clamp_min(1)[:, None], me)
                new = (q[:, :1] * me + al[:, None] * avg) / (q[:, 0] + al)[:, None]
                full[act] = torch.where(live[:, None], new, me)
        v, C = sc.g2p(full, cell, W, d)
        del full, cell, W, d
        damp = [torch.where(viscous, torch.exp(-rows[:, c].clamp_min(0) * dt), torch.ones_like(jp)) for c in (5, 6)]
        v, C = v * damp[0][:, None], C * damp[1][:, None, None]
        x = x + dt * v
        lo, hi = sc.p_origin + 2 * sc.p_dx[:, None], sc.p_origin + ((sc.p_G - 3) * sc.p_dx)[:, None]
        v = torch.where((x < lo) | (x > hi), torch.zeros_like(v), v)
        x = torch.minimum(torch.maximum(x, lo), hi)
        F = F + dt * _mm(C, F)
        root = (F[:, 0] * torch.linalg.cross(F[:, 1], F[:, 2])).sum(1).pow(1.0 / 3.0).clamp(0.05, 20.0)
        if some["solid"]:
            U, s0, V = _svd(F)
            s = s0
            if some["snow"]:
                s = torch.where(snow[:, None], torch.minimum(torch.maximum(s0, 1 - rows[:, 2:3]), 1 + rows[:, 3:4]), s)
                grown = (jp + torch.log(s0.prod(1).clamp_min(1e-6)) - torch.log(s.prod(1).clamp_min(1e-6))).clamp(-5, 5)
                jp = torch.where(snow, grown, jp)
            if some["sand"]:
                e = torch.log(s0.clamp_min(1e-6))
                tr = e.sum(1)
                dev_e = e - tr[:, None] / 3
                dn = dev_e.norm(dim=1)
                kappa = (3 * lam + 2 * mu) / (2 * mu)
                fy = dn + kappa * tr * rows[:, 1]
                out, slip = tr > 0, (tr <= 0) & (dn != 0) & (fy > 0)
                rc = (-rows[:, 1] * kappa * tr).clamp_min(0) / torch.where(dn > 0, dn, torch.ones_like(dn))
                back = torch.exp(dev_e * rc[:, None] + tr[:, None] / 3)
                s = torch.where((sand & slip)[:, None], back, torch.where((sand & out)[:, None], torch.ones_like(s), s))
                dq = torch.where(out, e.norm(dim=1), torch.where(slip, fy, torch.zeros_like(fy)))
                jp = torch.where(sand, (jp + dq).clamp(0, 5), jp)
            s = s.clamp(0.05, 20.0)
            F = _mm(U * s[:, None], V.transpose(1, 2))
        if bool(fluid.any()):
            s = torch.where(fluid[:, None], root[:, None], s)
            U = torch.where(fluid[:, None, None], I3, U)
            F = torch.where(fluid[:, None, None], root[:, None, None] * I3, F)
    return x, v, F, wrench


def _identify_run(cfgs, counts, x, v, E, F, dt, steps, target):
    """Forward and reverse-mode gradients of the differentiable model."""
    dev = _device()
    f32 = lambda a: torch.as_tensor(np.asarray(a, np.float32)).to(dev).to(torch.float64)  # noqa: E731
    sc = _Scenes(cfgs, counts)
    n = len(x)
    m = f32([c.particle_mass for c in cfgs])[sc.sid]
    vol = f32([c.particle_volume for c in cfgs])[sc.sid]
    nu = sc.nu[sc.sid]
    dt = float(np.float32(dt))
    x0, v0, E0 = (f32(t).requires_grad_() for t in (x, v, E))
    mu = E0 / (2 * (1 + nu))
    lam = E0 * nu / ((1 + nu) * (1 - 2 * nu))
    mu.retain_grad()
    lam.retain_grad()
    I3 = torch.eye(3, dtype=torch.float64, device=dev)

    def inv_t(R):  # inverse transpose: cofactors over the determinant
        a, b, c = R[:, 0], R[:, 1], R[:, 2]
        cof = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], 1)
        return cof / (a * cof[:, 0]).sum(1)[:, None, None]

    def substep(x, v, C, F, mu, lam):
        R = F
        for _ in range(6):  # Newton's iteration for the rotation of F
            R = 0.5 * (R + inv_t(R))
        tr = (R * F).sum((1, 2)) - 3
        P = 2 * mu[:, None, None] * (F - R) + (lam * tr)[:, None, None] * R
        A = m[:, None, None] * C - (dt * vol * 4 / sc.p_dx ** 2)[:, None, None] * _mm(P, F.transpose(1, 2))
        cell, W, d = sc.stencil(x)
        used, at = torch.unique(cell, return_inverse=True)
        mom = m[:, None, None] * v[:, None] + sum(A[:, None, :, j] * d[..., j, None] for j in range(3))
        q = torch.cat([(W * m[:, None])[..., None], W[..., None] * mom], -1).reshape(-1, 4)
        q = torch.zeros((len(used), 4), dtype=torch.float64, device=dev).index_add(0, at.reshape(-1), q)
        si, _, iy, _ = sc.where(used)
        gv = q[:, 1:] / q[:, :1]
        gx, gy, gz = gv[:, 0], gv[:, 1] + sc.gravity[si] * dt, gv[:, 2]
        under = sc.origin[si, 1] + iy * sc.dx[si] < sc.floor_y[si]
        damp = torch.where(under, 1 - sc.floor_friction[si], torch.ones_like(gx))
        gv = torch.stack([gx * damp, torch.where(under & (gy < 0), torch.zeros_like(gy), gy), gz * damp], 1)
        v, C = sc.g2p(gv, at, W, d)
        return x + dt * v, v, C, F + dt * _mm(C, F)

    s = (x0, v0, torch.zeros((n, 3, 3), dtype=torch.float64, device=dev), f32(F).reshape(n, 3, 3))
    for _ in range(steps):
        s = checkpoint(substep, *s, mu, lam, use_reentrant=False)
    xT = s[0]
    xT.backward((xT.detach() - target.to(torch.float64)))
    return {"x": xT.detach(), "gx": x0.grad, "gv": v0.grad, "gE": E0.grad,
            "gml": torch.stack([mu.grad.sum(), lam.grad.sum()])}


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 11])
    if kind == "keys":
        return None  # whole numbers
    if kind == "frame":
        if case["material"] == "large":
            cfg, d, _ = workloads.large_scene(case["particles"], seed=seed, grid=case["grid"])
            x, v, F, _ = _shader_run([cfg], [len(d["x"])], d["x"], d["v"], case["dt"], case["substeps"], d["mass"],
                                     d["volume"], d["material"])
        else:
            cfg, px, pv, mat = _box(case, rng)
            x, v, F, _ = _shader_run([cfg], [len(px)], px, pv, case["dt"], case["substeps"], mat=mat)
        return {"position": x, "velocity": v, "F": F.reshape(-1, 9)}
    if kind == "wheel":
        cfg, px, pv, wheel = _wheel_scene(case, rng)
        x, v, _, wrench = _shader_run([cfg], [len(px)], px, pv, 1e-4, case["substeps"], body=wheel)
        return {"wrench": wrench, "position": x, "velocity": v}
    if kind in ("batch", "rollouts"):
        cfgs, xs, vs, dt = _batch_scenes(case, seed)
        x, v, _, _ = _shader_run(cfgs, [len(p) for p in xs], np.concatenate(xs), np.concatenate(vs), dt,
                                 case["substeps"])
        return {"position": x, "velocity": v}
    cfgs, xs, vs, E, F, dt = _identify_scenes(case, seed)
    x = np.concatenate(xs)
    target = torch.from_numpy(_target(x)).to(_device())
    return _identify_run(cfgs, [len(p) for p in xs], x, np.concatenate(vs), E, F, dt, case["substeps"], target)

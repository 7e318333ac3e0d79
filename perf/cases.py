"""Timed workloads of the block-lattice backend: what a user's program has it do.

A pass is one stretch of a simulation between two outputs: time steps through
``collide_and_stream`` (a block, a split block, an ensemble, the solve server)
and then the result a program reads there: the fields its VTK writer takes
(``vtk.SuperLattice*3D``), the FP64 moments, or the solves' moments.  The state
goes on from pass to pass, as a simulation does.

The sizes are those of bench.py's workloads (256^3 porous channel, 384x192x192
turbulent channel, 201^3 benchmark cavity, cavities of 16-96 cells on an edge,
channel solves of 24-128) and smaller, odd and ragged ones of the same kinds.

``run`` calls only the public front end; ``exact`` is the same physics in plain
torch, FP64, without the package's kernels (the workload generators give both
sides the same geometry and initial state).
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from openlb_amd import serving, vtk, workloads
from openlb_amd.ensemble import Ensemble
from openlb_amd.lattice import BlockLattice
from openlb_amd.super_lattice import SuperLattice

BYTES = {"f64": 8, "f32": 4, "f16": 2}


def listed():
    return [
        # the headline workload: flow through a porous block, one output per 400 steps
        dict(name="porous_256_f32", kind="porous", nx=256, ny=256, nz=256, storage="f32", steps=400),
        # the same flow in FP64 on a ragged block
        dict(name="porous_odd_f64", kind="porous", nx=203, ny=131, nz=157, storage="f64", steps=200),
        # large-eddy channel in FP16 storage at the benchmark's size
        dict(name="turbulent_384_f16", kind="turbulent", nx=384, ny=192, nz=192, storage="f16", steps=300),
        # the same channel at a user's coarser, odd resolution in FP32
        dict(name="turbulent_odd_f32", kind="turbulent", nx=149, ny=97, nz=101, storage="f32", steps=400),
        # fully periodic vortex decay in FP64, evaluated as FP64 moments
        dict(name="tgv_128_f64", kind="tgv", q=19, nx=128, ny=128, nz=128, storage="f64", steps=300),
        # a small periodic D3Q27 box: launches and latency count
        dict(name="tgv_48_q27_f32", kind="tgv", q=27, nx=48, ny=48, nz=48, storage="f32", steps=300),
        # OpenLB's benchmark cavity, driven one collideAndStream() at a time as its harness does
        dict(name="cavity_local_201_f32", kind="cavity_local", n=201, storage="f32", steps=200),
        # the same cavity split into 2x2x2 cuboids on one device
        dict(name="cavity_split_101_f32", kind="cavity_split", n=101, blocks=2, storage="f32", steps=100),
        # uncertainty quantification: uneven cavities in FP16, replayed from a graph
        dict(name="ensemble_96_f16", kind="ensemble", members=96, lo=16, hi=96, storage="f16", steps=256, graph=True),
        # a handful of FP32 samples, stepped directly
        dict(name="ensemble_12_f32", kind="ensemble", members=12, lo=16, hi=64, storage="f32", steps=300, graph=False),
        # the solve server on a backlog of channel requests in both storages
        dict(name="serving_16", kind="serving", requests=16, lo=24, hi=96, steps_lo=200, steps_hi=800),
        # the smallest: a 24^3 cavity whose program reads the statistics every 10 steps
        dict(name="cavity_24_f32", kind="cavity_small", nx=24, ny=24, nz=24, storage="f32", steps=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["porous", "porous", "turbulent", "turbulent", "tgv", "tgv", "cavity_local", "cavity_split",
                       "ensemble", "ensemble", "serving", "cavity_small"])
    storage = rng.choice(["f32", "f32", "f16", "f64"])
    if kind == "porous":
        while True:
            n = [_log_int(rng, 32, 400) for _ in range(3)]
            if n[0] * n[1] * n[2] * BYTES[storage] <= 4 * 2 ** 24:
                break
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], storage=storage, steps=rng.randint(50, 400))
    if kind == "turbulent":
        while True:
            n = [_log_int(rng, 32, 400) for _ in range(3)]
            if n[0] * n[1] * n[2] * BYTES[storage] <= 2 * 2 ** 24:
                break
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], storage=storage, steps=rng.randint(50, 400))
    if kind == "tgv":
        while True:
            n = [_log_int(rng, 24, 256) for _ in range(3)]
            if n[0] * n[1] * n[2] * BYTES[storage] <= 2 ** 24:
                break
        return dict(kind=kind, q=rng.choice([19, 27]), nx=n[0], ny=n[1], nz=n[2], storage=storage,
                    steps=rng.randint(50, 300))
    if kind == "cavity_local":
        return dict(kind=kind, n=_log_int(rng, 32, 201), storage=rng.choice(["f32", "f64"]), steps=rng.randint(50, 200))
    if kind == "cavity_split":
        return dict(kind=kind, n=_log_int(rng, 24, 101), blocks=2, storage=rng.choice(["f32", "f64"]),
                    steps=rng.randint(20, 100))
    if kind == "ensemble":
        return dict(kind=kind, members=_log_int(rng, 4, 96), lo=16, hi=_log_int(rng, 40, 96), storage=storage,
                    steps=rng.randint(64, 256), graph=rng.random() < 0.5)
    if kind == "serving":
        return dict(kind=kind, requests=rng.randint(4, 16), lo=24, hi=rng.randint(48, 96), steps_lo=100, steps_hi=rng.randint(200, 800))
    n = [_log_int(rng, 12, 48) for _ in range(3)]
    return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], storage=storage, steps=10 * rng.randint(4, 12))


# ---- geometry and initial state ----------------------------------------------

def _cases(case, seed):
    """The workload (a list for an ensemble) that `seed` gives."""
    rng = np.random.Generator(np.random.PCG64(seed))
    kind = case["kind"]
    if kind == "porous":
        # spheres of radius 3-6 where they fit, a developed-looking start
        shape = (case["nx"], case["ny"], case["nz"])
        c = workloads.porous_channel(shape, seed=seed, force=1e-5)
        y, z = (np.arange(n, dtype=np.float64) for n in shape[1:])
        prof = (np.sin(np.pi * y / (shape[1] - 1))[:, None] * np.sin(np.pi * z / (shape[2] - 1))[None, :])
        c.rho_u[1] = float(rng.uniform(0.01, 0.02)) * prof[None]
        return c
    if kind == "turbulent":
        return workloads.turbulent_channel((case["nx"], case["ny"], case["nz"]), seed=seed,
                                           u_max=float(rng.uniform(0.04, 0.06)))
    if kind == "tgv":
        return workloads.taylor_green((case["nx"], case["ny"], case["nz"]), u0=float(rng.uniform(0.03, 0.06)),
                                      tau=float(rng.uniform(0.55, 0.8)), q=case["q"])
    if kind in ("cavity_local", "cavity_split"):
        n = case["n"]
        return workloads.local_velocity_cavity((n, n, n), tau=0.5 + 3.0e-5 * (n - 1) + 0.02,
                                               lid_u=float(rng.uniform(0.008, 0.012)))
    if kind == "cavity_small":
        return workloads.lid_driven_cavity((case["nx"], case["ny"], case["nz"]), tau=float(rng.uniform(0.55, 0.7)),
                                           lid_u=float(rng.uniform(0.03, 0.07)))
    if kind == "ensemble":
        # the study's extents are the case's own, its samples the seed's; tau
        # from 0.53, the lower bound of the FP16 precision guard
        shapes = workloads.cavity_ensemble(case["members"], lo=case["lo"], hi=case["hi"])
        return [workloads.lid_driven_cavity(m.shape, tau=float(rng.uniform(0.53, 1.2)), lid_u=float(rng.uniform(0.02, 0.1)))
                for m in shapes]
    raise ValueError(kind)


@dataclasses.dataclass
class _State:
    case: dict
    obj: object
    members: list
    requests: list

    def __del__(self):
        if self.obj is not None:
            self.obj.close()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serving":
        # the backlog's sizes, step counts and storages are the case's own, the inflow velocities the seed's
        rng = np.random.Generator(np.random.PCG64(seed))
        stream = serving.poisson_channel_stream(count=case["requests"], size=(case["lo"], case["hi"]),
                                                steps=(case["steps_lo"], case["steps_hi"]))
        reqs = [serving.channel_request(r.rid, r.arrival, r.case.shape[0], r.steps, float(rng.normal(0.05, 0.01)),
                                        r.storage) for r in stream]
        need = {"f32": 0, "f16": 0}
        for r in reqs:
            need[r.storage] += Ensemble.bytes_for(19, r.storage, r.case.shape)[0]
        srv = serving.SolveServer(budget_bytes=int(2.2 * max(need.values())), max_members=case["requests"],
                                  keep_moments=True)
        return _State(case, srv, [], reqs)
    c = _cases(case, seed)
    if kind == "ensemble":
        need = [Ensemble.bytes_for(19, case["storage"], m.shape) for m in c]
        ens = Ensemble(19, case["storage"], "bgk", max_members=len(c),
                       population_bytes=sum(n[0] for n in need) + (1 << 20),
                       cell_capacity=sum(n[1] for n in need) + (1 << 20))
        members = [ens.add(m) for m in c]
        for i, m in zip(members, c):
            ens.ini_equilibrium(i, m.rho_u)
        return _State(case, ens, members, [])
    if kind == "cavity_split":
        obj = SuperLattice(c, case["storage"], (case["blocks"],) * 3)
    else:
        obj = BlockLattice.from_case(c, case["storage"])
    obj.ini_equilibrium(c.rho_u)
    if c.local:
        obj.initialize()
    return _State(case, obj, [], [])


def _fields(lat):
    return {"density": vtk.SuperLatticeDensity3D(lat).evaluate(), "velocity": vtk.SuperLatticeVelocity3D(lat).evaluate()}


def run(state):
    case, obj = state.case, state.obj
    kind, steps = case["kind"], case.get("steps")
    if kind in ("porous", "turbulent"):
        obj.collide_and_stream(steps)
        return _fields(obj)
    if kind == "tgv":
        obj.collide_and_stream(steps)
        m = obj.moments()
        return {"density": m[0], "velocity": m[1:]}
    if kind == "cavity_local":
        for _ in range(steps):
            obj.collide_and_stream()
        return _fields(obj)
    if kind == "cavity_split":
        obj.collide_and_stream(steps)
        return {"density": [f.evaluate() for _, f in vtk.SuperLatticeDensity3D(obj).pieces()],
                "velocity": [f.evaluate() for _, f in vtk.SuperLatticeVelocity3D(obj).pieces()]}
    if kind == "cavity_small":
        stats = []
        for _ in range(0, steps, 10):
            for _ in range(10):
                obj.collide_and_stream()
            s = obj.statistics()
            stats.append([s["average_rho"], s["average_energy"], s["max_u"]])
        return {"statistics": np.array(stats), **_fields(obj)}
    if kind == "ensemble":
        obj.step(steps, graph=case["graph"])
        return np.concatenate([vtk.SuperLatticeVelocity3D(obj, member=m).evaluate(0) for m in state.members])
    results = sorted(obj.run(state.requests, realtime=False), key=lambda r: r.rid)
    return np.concatenate([r.moments.reshape(-1) for r in results])


# ---- what a pass cannot do without ---------------------------------------------

def work(case):
    """Every time step takes the state before it to the state after it: each
    population read once and written once per step, one id byte per cell where
    ids differ, plus the fields read out at the end.  About 12 flops per
    population and cell in a collision."""
    kind = case["kind"]
    if kind == "serving":
        # the mean request of the stream: log-uniform edge, half the requests in FP16
        lo, hi = case["lo"], case["hi"]
        cells = (hi ** 3 - lo ** 3) / (3.0 * math.log(hi / lo)) * case["requests"]
        steps = (case["steps_lo"] + case["steps_hi"]) / 2
        return {"bytes": cells * (steps * (2 * 19 * 3 + 1) + 32), "flops": cells * steps * 19 * 12}
    q = case["q"] if kind == "tgv" else (27 if kind == "turbulent" else 19)
    if kind == "ensemble":
        edge = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        cells, out = edge ** 3 * case["members"], 12
    elif "n" in case:
        cells, out = case["n"] ** 3, 16
    else:
        cells, out = case["nx"] * case["ny"] * case["nz"], 32 if kind == "tgv" else 16
    ids = 0 if kind == "tgv" else 1
    return {"bytes": float(cells * (case["steps"] * (2 * q * BYTES[case["storage"]] + ids) + out)),
            "flops": float(cells * case["steps"] * q * 12)}


def tolerance(case):
    """About four times the largest error measured against `exact` over the
    listed and thirty drawn cases: FP64 moments 3e-15, float32 fields of an
    FP64 lattice 2.6e-8, velocities of FP32 lattices 1.6e-5 and of FP16
    lattices 5.5e-4 (every population of a slow flow is rounded once per step).
    The solves' moments hold density and velocity side by side."""
    kind = case["kind"]
    if kind == "serving":
        return {"rel": 1e-4}
    if case["storage"] == "f64":
        return {"rel": 2e-14 if kind == "tgv" else 1e-7}
    return {"rel": 6.4e-5 if case["storage"] == "f32" else 2.2e-3}


# ---- the same physics in plain torch, FP64 --------------------------------------

def _velocities(q):
    """Discrete velocities and weights of D3Q19 / D3Q27 (any order: only sums leave)."""
    c, w = [], []
    by_norm = {19: {0: 1 / 3, 1: 1 / 18, 2: 1 / 36}, 27: {0: 8 / 27, 1: 2 / 27, 2: 1 / 54, 3: 1 / 216}}[q]
    for x in (-1, 0, 1):
        for y in (-1, 0, 1):
            for z in (-1, 0, 1):
                n = x * x + y * y + z * z
                if n in by_norm:
                    c.append((x, y, z))
                    w.append(by_norm[n])
    return c, w


def _equilibrium(c, w, rho, u, out):
    """f_i - w_i of the second-order equilibrium."""
    base = 1 - 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    for i, (ci, wi) in enumerate(zip(c, w)):
        feq = base.clone()
        if any(ci):
            cu = sum(u[d] * ci[d] for d in range(3) if ci[d])
            feq.add_(cu, alpha=3).addcmul_(cu, cu, value=4.5)
        out[i] = feq.mul_(rho).sub_(1).mul_(wi)


def _moments(c, f):
    rho = f.sum(0) + 1
    u = []
    for d in range(3):
        j = torch.zeros_like(rho)
        for i, ci in enumerate(c):
            if ci[d]:
                j.add_(f[i], alpha=ci[d])
        u.append(j / rho)
    return rho, u


class _Plain:
    """Collide, then stream on the periodic box, for any number of blocks side
    by side in one flat array.  What leaves through a wall face comes in at the
    other side, into wall cells, which send it back: it never meets the fluid."""

    def __init__(self, cases):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.cases, first = cases, cases[0]
        self.kind, self.force = first.kind, first.force
        self.c, self.w = _velocities(first.q)
        self.opp = [self.c.index(tuple(-x for x in ci)) for ci in self.c]
        self.start = np.cumsum([0] + [m.ncore for m in cases])
        n = int(self.start[-1])
        self.ids = torch.cat([torch.from_numpy(m.ids).to(dev).reshape(-1) for m in cases])
        self.bulk = self.ids == 1
        self.all_bulk = bool(self.bulk.all())
        self.forced = first.kind == "forced_bgk"
        self.tau = 1.0 / first.omega
        if len(cases) > 1:
            self.tau = torch.cat([torch.full((m.ncore,), 1.0 / m.omega, dtype=torch.float64, device=dev) for m in cases])
        # moving walls: cells, fixed density and velocity
        self.walls = []
        for m, lo in zip(cases, self.start):
            for wid, (rw, uw) in m.walls.items():
                at = torch.from_numpy(np.flatnonzero(m.ids == wid) + lo).to(dev)
                self.walls.append((at, rw, uw))
        # pull[i][cell]: the cell whose i-th population arrives here
        self.pull = torch.empty((len(self.c), n), dtype=torch.int32, device=dev)
        for m, lo in zip(cases, self.start):
            x, y, z = (torch.arange(k, dtype=torch.int32, device=dev) for k in m.shape)
            nx, ny, nz = m.shape
            for i, ci in enumerate(self.c):
                sx, sy, sz = (x - ci[0]) % nx, (y - ci[1]) % ny, (z - ci[2]) % nz
                src = (sx[:, None, None] * ny + sy[None, :, None]) * nz + sz[None, None, :] + int(lo)
                self.pull[i, lo:lo + m.ncore] = src.reshape(-1)
        rho_u = [torch.cat([torch.from_numpy(m.rho_u[d]).to(dev).reshape(-1) for m in cases]) for d in range(4)]
        u = rho_u[1:]
        if self.forced:
            u = [u[d] - 0.5 * self.force[d] * self.bulk for d in range(3)]
        self.f = torch.empty((len(self.c), n), dtype=torch.float64, device=dev)
        _equilibrium(self.c, self.w, rho_u[0], u, self.f)
        self.g = torch.empty_like(self.f)

    def moments(self):
        rho, u = _moments(self.c, self.f)
        if self.forced:
            u = [u[d] + 0.5 * self.force[d] for d in range(3)]
        return rho, u

    def omega(self, rho, u):
        tau = self.tau
        if self.kind != "smagorinsky":
            return 1.0 / tau
        # |Pi_neq| from the second moments about the equilibrium
        norm = torch.zeros_like(rho)
        for a in range(3):
            for b in range(a, 3):
                p = -rho * u[a] * u[b]
                for i, ci in enumerate(self.c):
                    if ci[a] * ci[b]:
                        p.add_(self.f[i], alpha=ci[a] * ci[b])
                if a == b:
                    p.sub_(rho - 1, alpha=1 / 3)
                norm.add_(p * p, alpha=1 if a == b else 2)
        norm.sqrt_()
        cs2 = 18 * math.sqrt(2.0) * self.cases[0].smago ** 2
        return 1.0 / (0.5 * tau + 0.5 * torch.sqrt(tau * tau + cs2 * norm / rho))

    def step(self):
        f, g = self.f, self.g
        rho, u = self.moments()
        om = self.omega(rho, u)
        _equilibrium(self.c, self.w, rho, u, g)
        if self.forced:
            uf = sum(u[d] * self.force[d] for d in range(3))
        for i, (ci, wi) in enumerate(zip(self.c, self.w)):
            g[i].sub_(f[i]).mul_(om).add_(f[i])
            if self.forced:
                cf = sum(ci[d] * self.force[d] for d in range(3))
                cu = sum(u[d] * ci[d] for d in range(3))
                g[i].add_(rho * (3 * cf + 9 * cu * cf - 3 * uf), alpha=wi * (1 - 0.5 / self.tau))
            if not self.all_bulk:
                g[i] = torch.where(self.bulk, g[i], f[self.opp[i]])
                for at, rw, uw in self.walls:
                    corr = 6 * rw * wi * sum(ci[d] * uw[d] for d in range(3))
                    if corr:
                        g[i, at] += corr
        for i in range(len(self.c)):
            torch.index_select(g[i], 0, self.pull[i], out=f[i])

    def cell_fields(self):
        """What each cell's own dynamics report: the moments of a bulk cell, a wall's fixed values."""
        rho, u = self.moments()
        full = torch.stack([rho] + u)
        if not self.all_bulk:
            full[0][~self.bulk] = 1
            full[1:, ~self.bulk] = 0
            for at, rw, uw in self.walls:
                for d, v in enumerate((rw,) + tuple(uw)):
                    full[d, at] = v
        return full

    def fields(self, overlap):
        """Per block, density and velocity in VTK point order (x fastest) with
        `overlap` cells around: periodic images of bulk cells, else rho 1 and u 0."""
        flat, out = self.cell_fields(), []
        for m, lo in zip(self.cases, self.start):
            full = flat[:, lo:lo + m.ncore].reshape((4,) + tuple(m.shape))
            bulk = self.bulk[lo:lo + m.ncore].reshape(m.shape)
            if overlap:
                idx, inside = [], torch.ones([n + 2 * overlap for n in m.shape], dtype=torch.bool, device=full.device)
                core = torch.ones_like(inside)
                for d, n in enumerate(m.shape):
                    r = torch.arange(-overlap, n + overlap, device=full.device)
                    view = [1, 1, 1]
                    view[d] = len(r)
                    at = ((r >= 0) & (r < n)).view(view)
                    core &= at
                    if not m.periodic[d]:
                        inside &= at
                    idx.append(r % n)
                sel = (idx[0][:, None, None], idx[1][None, :, None], idx[2][None, None, :])
                rest = torch.tensor([1.0, 0, 0, 0], dtype=full.dtype, device=full.device).view(4, 1, 1, 1)
                full = torch.where(inside & (core | bulk[sel]), full[(slice(None),) + sel], rest)
            full = full.permute(0, 3, 2, 1)
            out.append({"density": full[0].reshape(-1).cpu().numpy(),
                        "velocity": full[1:].permute(1, 2, 3, 0).reshape(-1).cpu().numpy()})
        return out

    def statistics(self):
        """Average density, average energy and largest speed over bulk cells and moving walls."""
        full = self.cell_fields()[:, (self.ids == 1) | (self.ids >= 3)]
        usq = full[1] ** 2 + full[2] ** 2 + full[3] ** 2
        return [float(full[0].mean()), 0.5 * float(usq.mean()), math.sqrt(float(usq.max()))]


def exact(case, seed):
    """None for the cavities and channels with LocalVelocity / LocalPressure
    boundaries: their reconstruction, cell type by cell type and from
    neighbouring velocities, has no short plain form."""
    kind, steps = case["kind"], case.get("steps")
    if kind in ("cavity_local", "cavity_split", "serving"):
        return None
    cells = case["members"] * 1e5 if kind == "ensemble" else case["nx"] * case["ny"] * case["nz"]
    if not torch.cuda.is_available() and cells * steps > 2e7:
        return None  # minutes on a CPU
    c = _cases(case, seed)
    p = _Plain(c if kind == "ensemble" else [c])
    stats = []
    for k in range(steps):
        p.step()
        if kind == "cavity_small" and (k + 1) % 10 == 0:
            stats.append(p.statistics())
    if kind == "ensemble":
        return np.concatenate([m["velocity"] for m in p.fields(0)])
    if kind == "tgv":
        rho, u = p.moments()
        return {"density": rho.reshape(c.shape).cpu().numpy(),
                "velocity": torch.stack(u).reshape((3,) + tuple(c.shape)).cpu().numpy()}
    if kind == "cavity_small":
        return {"statistics": np.array(stats), **p.fields(1)[0]}
    return p.fields(1)[0]

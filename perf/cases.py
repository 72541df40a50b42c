"""The work that programs have this library do, as timed passes through its public Python API.

Three kinds of pass:

* "step"  — one batch of an SPH run: stepsolve_ over `steps` adaptive steps of one problem (or batch_stepsolve_ of an
            ensemble), then the state is read back, as a monitoring, coupling or output loop does (timesolve_ is that
            loop).  The scenes are the dam breaks of the tests, the benchmark and `gclsph.scenes`, in motion: a smooth
            velocity field and a small disorder of the lattice, both from the seed.
* "list"  — the cell list on its own: the points have moved, update_ (or partialupdate_) and the pair list.
* "device" — neighborlist_noalloc on coordinates and a pair buffer that live on the GPU.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpucelllistsph.jl_amd"))

import gclsph as G  # noqa: E402
from gclsph import scenes as S  # noqa: E402


def listed():
    def step(name, dim, precision, dx, width, height, tank, steps, walls="fixture", factor=1.0, physics="base", scenes=1):
        return {"name": name, "kind": "step", "dim": dim, "precision": precision, "dx": dx, "width": width,
                "height": height, "tank": tank, "steps": steps, "walls": walls, "factor": factor, "physics": physics,
                "scenes": scenes}

    def points(name, kind, dim, precision, n, dist, call="update"):
        return {"name": name, "kind": kind, "dim": dim, "precision": precision, "n": n, "dist": dist, "call": call}

    return [
        # the smallest call: one step (stepsolve_'s default) of the tests' small scene, e.g. coupled to another solver
        step("step2d-0.5k-f64", 2, "f64", 0.05, 0.5, 1.0, 2.0, 1, walls="minus1"),
        # the 2D dam break of 5,000 fluid particles in timesolve_'s default batches of ten steps
        step("step2d-6k-f64", 2, "f64", 0.02, 1.0, 2.0, 4.0, 10, walls="minus1"),
        # a small run with the reference examples' dist = 1.1 H: most steps keep the neighbour lists
        step("step2d-25k-f32split", 2, "f32split", 0.0105, 1.3, 1.9, 4.0, 50, factor=1.1),
        # an ordinary run in Float64, lists kept over steps, uneven sizes
        step("step2d-250k-f64", 2, "f64", 0.0041, 1.97, 2.03, 8.0, 30, factor=1.1),
        # a large run in Float64, rebuilding every step
        step("step2d-1M-f64", 2, "f64", 0.004, 4.0, 4.0, 16.0, 40),
        # the benchmark's scene: 4,000,000 fluid particles, FP32-split, a frame every hundred steps
        step("step2d-4M-f32split", 2, "f32split", 0.002, 4.0, 4.0, 16.0, 100),
        # 3D in Float64 with every physics term (viscosity, surface tension, DPC, XSPH, CSPM), small
        step("step3d-32k-f64-all", 3, "f64", 0.04, 1.0, 1.0, 3.2, 10, walls="minus1", physics="all"),
        # 3D in Float64, the terms that are on by default, dist = 1.1 H
        step("step3d-191k-f64", 3, "f64", 0.0185, 1.0, 1.0, 3.2, 10, factor=1.1),
        # the benchmark's 3D scene (883,376 particles), FP32-split, every physics term
        step("step3d-880k-f32split-all", 3, "f32split", 0.01, 1.0, 1.0, 3.2, 20, walls="minus1", physics="all"),
        # the ensemble: 64 dam breaks of 1,500 to 120,000 particles stepped together
        step("ensemble-64-f32split", 2, "f32split", 0.0, 0.0, 0.0, 4.0, 30, scenes=64),
        # the reference's own cell-list benchmark: 200,000 uniform points, 79 pairs per point
        points("list2d-200k-f64", "list", 2, "f64", 200_000, 0.016),
        # neighbour lists for a program that keeps its data on the GPU and must not allocate
        points("device3d-300k-f64", "device", 3, "f64", 300_007, 0.026),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(("step", "step", "step", "step", "list", "device"))
    if kind != "step":
        dim = rng.choice((2, 3))
        n = int(log(2_000, 500_000))
        around = log(12, 120)  # neighbours per point, either side
        dist = (around / (n * (math.pi if dim == 2 else 4 / 3 * math.pi))) ** (1 / dim)
        return {"kind": kind, "dim": dim, "precision": rng.choice(("f64", "f32")) if kind == "list" else "f64", "n": n,
                "dist": dist, "call": rng.choice(("update", "partialupdate")) if kind == "list" else "update"}
    dim = rng.choice((2, 2, 3))
    precision = rng.choice(("f64", "f32split"))
    width, height = rng.uniform(0.7, 1.5), rng.uniform(0.8, 2.0) if dim == 2 else rng.uniform(0.5, 1.0)
    n = log(700, 1_500_000) if dim == 2 else log(4_000, 300_000)
    dx = (width * height * (1.0 if dim == 2 else 0.5) / n) ** (1 / dim)
    most = 60 if n < 100_000 else 30
    return {"kind": "step", "dim": dim, "precision": precision, "dx": dx, "width": width, "height": height,
            "tank": rng.uniform(2.5, 4.0), "steps": rng.randint(1, most if dim == 2 else most // 3),
            "walls": rng.choice(("minus1", "fixture")) if dim == 2 else "minus1", "factor": rng.choice((1.0, 1.1, 1.2)),
            "physics": rng.choice(("base", "all")), "scenes": 1}


# ------------------------------------------------------------------ scenes
@functools.lru_cache(maxsize=80)
def lattice(dim, dx, width, height, tank, walls):
    """Fluid column and three wall layers on the lattice of `gclsph.scenes`: (points, ptype, fluid count)."""
    if dim == 3:
        depth = 0.5
        nf = [int(round(a / dx)) for a in (width, height, depth)]
        ext = [max(tank, (nf[0] + 5) * dx), 1.5, (nf[2] + 5) * dx]
        f = [3 * dx + dx * np.arange(n) for n in nf]
        fluid = [a.ravel() for a in np.meshgrid(*f, indexing="ij")]
        g = [a.ravel() for a in np.meshgrid(*(dx * np.arange(int(round(e / dx)) + 1) for e in ext), indexing="ij")]
        lay = 2.5 * dx
        shell = (g[1] < lay) | (g[0] < lay) | (g[0] > ext[0] - lay) | (g[2] < lay) | (g[2] > ext[2] - lay)
        wall = [a[shell] for a in g]
        wt = np.full(wall[0].size, -1, np.int32)
        if walls == "fixture":  # the layer next to the fluid takes part in density and pressure
            near = 1.5 * dx
            out = ((wall[1] < near) | (wall[0] < near) | (wall[0] > ext[0] - near) | (wall[2] < near) |
                   (wall[2] > ext[2] - near))
            wt = np.where(out, 0, 1).astype(np.int32)
    else:
        nf = [int(round(a / dx)) for a in (width, height)]
        ext = [max(tank, (nf[0] + 5) * dx), max(3.0 if tank < 5 else tank / 2, (nf[1] + 5) * dx)]
        fluid = [a.ravel() for a in np.meshgrid(*(3 * dx + dx * np.arange(n) for n in nf), indexing="ij")]
        wall = list(S.tank_boundary_2d(dx, *ext))
        wt = np.full(wall[0].size, -1, np.int32)
        if walls == "fixture":
            wt = S.fixture_wall_types(wall[0], wall[1], dx, int(round(ext[0] / dx)) * dx)
    points = tuple(np.concatenate([a, b]) for a, b in zip(fluid, wall))
    return points, np.concatenate([np.full(fluid[0].size, 2, np.int32), wt]), fluid[0].size


def scene(case, seed):
    """Points, velocities, densities, types, parameters and dist of a "step" case's scene."""
    dim, dx = case["dim"], case["dx"]
    points, ptype, nf = lattice(dim, dx, case["width"], case["height"], case["tank"], case["walls"])
    p, dist = S.standard_params(dx, dim, dist_factor=case["factor"])
    if case["physics"] == "all":
        p.nu, p.s, p.dpc_l0, p.dpc_lambda, p.dpc_pmax, p.xsph_eps = 0.2, 0.05, 0.5 * dx, 0.005, 36000.0, 0.5
    rng = np.random.default_rng(seed)
    points = [a.copy() for a in points]
    v = [np.zeros(a.size) for a in points]
    rho = np.full(ptype.size, p.rho0)
    y = points[1][:nf]
    rho[:nf] = S.hydrostatic_rho(y, y.max(), p.rho0, p.g, p.c0)
    # a divergence-free roll in (x, y) of about half a metre per second and, in 3D, a drift along z
    kx, ky = (2 * math.pi * rng.uniform(0.6, 1.4) / a for a in (case["width"], case["height"]))
    ax, ay = kx * points[0][:nf] + rng.uniform(0, 2 * math.pi), ky * y + rng.uniform(0, 2 * math.pi)
    amp = rng.uniform(0.3, 0.6)
    v[0][:nf] = amp * np.sin(ax) * np.cos(ay)
    v[1][:nf] = -amp * kx / ky * np.cos(ax) * np.sin(ay)
    if dim == 3:
        v[2][:nf] = 0.1 * np.cos(ax)
    for a in points:
        a[:nf] += 0.004 * dx * (rng.random(nf) - 0.5)
    return points, v, rho, ptype, p, dist


def members(case, seed):
    """The scenes of a "step" case: itself, or the seeded ensemble (the ranges of gclsph.scenes.config4)."""
    if case["scenes"] == 1:
        return [scene(case, seed)]
    u = [S.uniform01(4, case["scenes"], k) for k in range(3)]
    return [scene({**case, "dx": (0.005, 0.01, 0.02)[min(int(u[0][i] * 3), 2)], "width": round(0.5 + float(u[1][i]), 2),
                   "height": round(1.0 + float(u[2][i]), 2)}, seed + 1000 * i) for i in range(case["scenes"])]


def cloud(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.random(case["n"]) for _ in range(case["dim"])], rng


# ------------------------------------------------------------------ passes
def prepare(case, seed):
    if case["kind"] == "step":
        problems = []
        for points, v, rho, ptype, p, dist in members(case, seed):
            cells = G.GPUCellList(points, (dist,) * case["dim"], dist)
            problems.append(G.SPHProblem.from_params(cells, p, rho, ptype, v=v, precision=case["precision"]))
        return {"case": case, "problems": problems, "batch": G.SPHBatch(problems) if case["scenes"] > 1 else None}
    points, rng = cloud(case, seed)
    dist = case["dist"]
    if case["kind"] == "list":
        cells = G.GPUCellList(points, (dist,) * case["dim"], dist, mpairs=int(1.1 * pairs_of(case)),
                              precision=case["precision"])
        moved = [a + rng.normal(0.0, min(0.001, dist / 16), a.size) for a in points]
        return {"case": case, "cells": cells, "moved": moved}
    return {"case": case, "x": [torch.from_numpy(a).cuda() for a in points],
            "pairs": torch.zeros(int(1.1 * pairs_of(case)), 2, dtype=torch.int32, device="cuda")}


def run(state):
    case = state["case"]
    if case["kind"] == "list":
        cells = state["cells"]
        cells.points = state["moved"]
        (G.update_ if case["call"] == "update" else G.partialupdate_)(cells)
        return G.neighborlist(cells), cells.pairsn
    if case["kind"] == "device":
        x, dim = state["x"], case["dim"]
        total = G.neighborlist_noalloc([a.data_ptr() for a in x], case["n"], (case["dist"],) * dim, case["dist"],
                                       (0.0,) * dim, (1.0,) * dim, state["pairs"].data_ptr(), state["pairs"].shape[0])
        return state["pairs"], total
    if state["batch"] is not None:
        updates, travel = G.batch_stepsolve_(state["batch"], case["steps"], timestepping=True)
    else:
        updates, travel = G.stepsolve_(state["problems"][0], case["steps"], timestepping=True)
    each = [read(p, case["precision"]) for p in state["problems"]]
    if len(each) == 1:
        x, v, rho = each[0]
    else:
        x, v = (tuple(np.concatenate([e[w][k] for e in each]) for k in range(case["dim"])) for w in (0, 1))
        rho = np.concatenate([e[2] for e in each])
    return {"x": x, "v": v, "rho": rho, "updates": updates, "travel": travel,
            "time": np.array([G.get_simtime(p) for p in state["problems"]])}


def read(problem, precision):
    x, v, rho = G.get_points(problem), G.get_velocity(problem), G.get_density(problem)
    if precision == "f32split":  # held in 32 bits: velocity, and density as its difference from the rest density
        return x, tuple(a.astype(np.float32) for a in v), (rho - problem.rho0).astype(np.float32)
    return x, v, rho


# ------------------------------------------------------------------ work
def pairs_of(case):
    """Expected pairs of a "list" or "device" case: two uniform points of the unit square or cube nearer than dist."""
    d, n = case["dist"], case["n"]
    if case["dim"] == 2:
        near = math.pi * d ** 2 - 8 / 3 * d ** 3 + d ** 4 / 2
    else:
        near = 4 / 3 * math.pi * d ** 3 - 1.5 * math.pi * d ** 4 + 1.6 * d ** 5 - d ** 6 / 6
    return n * (n - 1) / 2 * near


def work(case):
    dim = case["dim"]
    if case["kind"] != "step":
        size = 4 if case["precision"] == "f32" else 8
        return {"bytes": case["n"] * dim * size + 8 * pairs_of(case), "flops": (3 * dim - 1) * pairs_of(case)}
    n = sum(m[3].size for m in members(case, 0)) if case["scenes"] > 1 else lattice(
        dim, case["dx"], case["width"], case["height"], case["tank"], case["walls"])[1].size
    word = 4 if case["precision"] == "f32split" else 8
    # each step reads and writes every particle's position, velocity and density; the state is handed out at the end
    per_step = 2 * n * (8 * dim + word * (dim + 1)) + 4 * n
    reach = case["factor"] * 2.4 * math.sqrt(2)
    half = n * (math.pi * reach ** 2 if dim == 2 else 4 / 3 * math.pi * reach ** 3) / 2
    # a pair once per evaluation: ~70 operations each in two evaluations, ~40 in each correction
    flops = half * (140 + (120 if case["physics"] == "all" else 0))
    return {"bytes": case["steps"] * per_step + n * (8 * dim + word * (dim + 1)), "flops": case["steps"] * flops}


# ------------------------------------------------------------------ the same in 64 bits
def exact(case, seed):
    """The pass in plain float64 torch: explicit pair lists, the equations of the step term by term."""
    if case["kind"] != "step":
        return None  # whole numbers
    got = members(case, seed)
    if sum(m[3].size for m in got) * (36 if case["dim"] == 2 else 160) * case["steps"] > 2.5e9:
        return None  # too long
    each = [Plain(case["dim"], *m).steps(case["steps"]) for m in got]
    x, v = ([torch.cat([e[w][k] for e in each]).cpu().numpy() for k in range(case["dim"])] for w in (0, 1))
    rho = torch.cat([e[2] for e in each]).cpu().numpy()
    if case["precision"] == "f32split":
        rho = rho - got[0][4].rho0
    return {"x": tuple(x), "v": tuple(v), "rho": rho, "updates": None,
            "travel": np.array([e[4] for e in each]) if len(each) > 1 else each[0][4], "time": np.array([e[3] for e in each])}


class Plain:
    """Weakly compressible SPH with the symplectic scheme of stepsolve_, over directed pairs (i, j) in float64."""

    def __init__(self, dim, points, v, rho, ptype, p, dist):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dim, self.p, self.dist = dim, p, dist
        self.x = torch.stack([torch.as_tensor(a) for a in points]).to(dev)
        self.v = torch.stack([torch.as_tensor(a) for a in v]).to(dev)
        self.rho = torch.as_tensor(rho).to(dev)
        self.pt = torch.as_tensor(ptype).to(dev)
        self.norm = 7 / math.pi if dim == 2 else 21 / (2 * math.pi)

    def W(self, u, H):
        return torch.where(u < 1, (1 - u) ** 4 * (1 + 4 * u), 0.0) * self.norm / H ** self.dim

    def pairs(self):
        """Directed pairs nearer than dist: points sorted into square cells, one row of three cells at a time."""
        x, d = self.x, self.dist
        c = ((x - x.amin(1, keepdim=True)) / d).floor().long() + 1
        size = c.amax(1) + 2
        key = c[-1]
        for k in range(self.dim - 2, -1, -1):
            key = key * size[k] + c[k]
        order = torch.argsort(key)
        skey = key[order]
        found = []
        for row in range(3 ** (self.dim - 1)):
            at = key + (row % 3 - 1) * size[0] + ((row // 3 - 1) * size[0] * size[1] if self.dim == 3 else 0)
            lo, hi = torch.searchsorted(skey, at - 1), torch.searchsorted(skey, at + 1, right=True)
            n = hi - lo
            i = torch.repeat_interleave(torch.arange(n.numel(), device=n.device), n)
            j = order[torch.arange(i.numel(), device=n.device) - (n.cumsum(0) - n)[i] + lo[i]]
            near = ((x[:, i] - x[:, j]).square().sum(0) < d * d) & (i != j)
            found.append((i[near], j[near]))
        self.i, self.j = (torch.cat([f[k] for f in found]) for k in (0, 1))

    def sum(self, terms):
        return torch.zeros_like(self.rho).index_add_(0, self.i, terms)

    def eos(self, rho):
        p = self.p
        P = p.c0 ** 2 * p.rho0 / p.gamma * ((rho / p.rho0) ** p.gamma - 1)
        return torch.where((self.pt <= 1) & (rho < p.rho0), 0.0, P)

    def rates(self, x, v, rho, grad, sep, r, bound):
        """(density rate, acceleration): grad is the kernel gradient, sep and r the separation of the wall force."""
        p, i, j = self.p, self.i, self.j
        dx, dv = x[:, i] - x[:, j], v[:, i] - v[:, j]
        ri, rj, ti, tj = rho[i], rho[j], self.pt[i], self.pt[j]
        r2 = dx.square().sum(0)
        den = r2 + (0.1 * p.h) ** 2
        both = (ti > 0) & (tj > 0)
        z = p.rho0 * p.g / (p.c0 ** 2 * p.rho0 / p.gamma) * dx[1]
        hydro = p.rho0 * torch.expm1(torch.log1p(z) / p.gamma)
        diffuse = 2 * p.h * p.delta * p.c0 * (rj - ri - hydro) / den * -(dx * grad).sum(0) * p.m0 / rj
        drho = self.sum(torch.where(both, p.m0 * (dv * grad).sum(0) + torch.where(ti > 1, diffuse, 0.0), 0.0))
        P = self.eos(rho)
        alike = both | ((ti < 0) & (tj < 0))
        along = torch.where(alike, -p.m0 * (P[i] + P[j]) / (ri * rj), 0.0)
        approach = (dv * dx).sum(0).clamp(max=0)
        along = along + torch.where(both, p.alpha * p.c0 * p.h * approach / den / ((ri + rj) / 2) * p.m0, 0.0)
        a = along * grad
        if p.nu > 0:
            a = a + torch.where(both, 4 * p.nu * p.m0 * (dx * grad).sum(0) / ((ri + rj) * den), 0.0) * dv
        if p.s > 0:
            now = r2.sqrt()
            pull = p.s * torch.cos(1.5 * math.pi * now / (2 * p.h)) / (now + 0.1 * p.h) / p.m0
            a = a + torch.where(both & (now < 2 * p.h), pull, 0.0) * dx
        D, r0 = bound
        q = r0 / (r + 0.01 * r0 ** 2)
        wall = ((ti > 0) != (tj > 0)) & (r < r0)
        a = a + torch.where(wall, D * (q ** 12 - q ** 4) / (r * r + 0.01 * r0 ** 2), 0.0) * sep
        acc = torch.stack([self.sum(a[k]) for k in range(self.dim)])
        acc[1] -= p.g
        return drho, acc

    def dpc(self, dt):
        """Velocity correction of close particles (dynamic particle collision)."""
        p, i, j = self.p, self.i, self.j
        dx, dv = self.x[:, i] - self.x[:, j], self.v[:, i] - self.v[:, j]
        r2 = dx.square().sum(0)
        u, den = r2.sqrt() / p.dpc_l0, r2 + (0.1 * p.dpc_l0) ** 2
        half = self.W(torch.tensor(0.5, dtype=torch.float64), p.dpc_l0)
        chi = (self.W(u, p.dpc_l0) / half).sqrt()
        lo, hi = 0.0, 1.0  # where the kernel of unit support falls to one
        for _ in range(100):
            mid = (lo + hi) / 2
            lo, hi = (mid, hi) if (1 - mid) ** 4 * (1 + 4 * mid) * self.norm > 1 else (lo, mid)
        P = self.eos(self.rho)
        push = (p.dpc_lambda * (P[i] + P[j]).abs()).clamp(max=p.dpc_lambda * p.dpc_pmax).clamp(min=p.dpc_pmin) * chi
        meet = (dv * dx).sum(0)
        k = torch.where(meet < 0, -torch.where(u < lo, 1.0, chi) * meet / den,
                        2 * dt * push / ((self.rho[i] + self.rho[j]) * den))
        k = torch.where((self.pt[i] > 0) & (self.pt[j] > 0), k, 0.0)
        return torch.stack([self.sum(k * dx[d]) for d in range(self.dim)])

    def steps(self, n):
        p, pt = self.p, self.pt
        dt, clock, travel, moved, rebuild = p.dt, 0.0, 0.0, torch.zeros_like(self.x), True
        limits = (math.sqrt(np.finfo(np.float64).eps), p.CFL * p.H / (3 * p.c0))
        before = (self.x, self.v, self.rho)  # the state before the last step's corrections: half steps start there
        for it in range(1, n + 1):
            if rebuild:
                self.pairs()
                moved, rebuild = torch.zeros_like(self.x), False
            i, j = self.i, self.j
            sep = self.x[:, i] - self.x[:, j]
            r = sep.square().sum(0).sqrt()
            u = r / p.H
            grad = torch.where(u < 1, -20 * (1 - u) ** 3, 0.0) * self.norm / p.H ** (self.dim + 2) * sep
            drho, acc = self.rates(self.x, self.v, self.rho, grad, sep, r, (0.4, 2 * p.dx))
            rho = before[2] + drho * dt / 2
            rho = torch.where((pt < 0) & (rho < p.rho0), p.rho0, rho)
            v = before[1] + torch.where(pt > 1, acc * dt / 2, 0.0)
            drho, acc = self.rates(before[0] + v * dt / 2, v, rho, grad, sep, r, (p.bound_D, p.bound_l))
            eps = -drho / rho * dt
            rho = self.rho * (2 - eps) / (2 + eps)
            rho = torch.where((pt <= 1) & (rho < p.rho0), p.rho0, rho)
            v = self.v + torch.where(pt > 1, acc * dt, 0.0)
            go = (self.v + v) / 2 * dt
            moved, start = moved + go, self.x
            self.x, self.v, self.rho = self.x + go, v, rho
            before = (self.x, self.v, self.rho)
            if p.dpc_l0 > 0:
                dv = torch.where(pt > 1, self.dpc(dt), 0.0)
                self.x, self.v = self.x + dv * dt, self.v + dv
            if p.xsph_eps > 0:
                w = 2 * p.m0 * p.xsph_eps * self.W(u, p.H) / (self.rho[i] + self.rho[j])
                w = torch.where((pt[i] > 1) & (pt[j] > 1), w, 0.0)
                drift = [self.sum(w * (self.v[d, j] - self.v[d, i])) for d in range(self.dim)]
                self.x = self.x + dt * torch.stack(drift)
            if it % p.cspmn == 0:
                w = torch.where((pt[i] > 0) & (pt[j] > 0), self.W(u, p.H), 0.0)
                new = self.sum(w) / self.sum(w / self.rho[j])
                self.rho = torch.where(new.isnan(), self.rho, new)
            far = float(moved.abs().max())
            rebuild, travel, clock = far > 0.9 * p.nui, max(travel, far), clock + dt
            fast = p.h * (self.v * self.x).sum(0) / (self.x.square().sum(0) + (0.01 * p.h) ** 2)
            force = float(acc.square().sum(0).max().sqrt())
            dt = p.CFL * min(math.sqrt(p.h / (3 * force)), p.h / (p.c0 + float(fast.abs().max())))
            dt = min(max(dt, limits[0]), limits[1])
        return self.x, self.v, self.rho, clock, travel

"""Measured workloads: the calls that a simulation program makes between two
outputs, through the package's Python driver (nlmech_amd.engine.GpuFD).

An explicit case advances a prepared model by the steps between two outputs
and reads back what an output holds: displacement, velocity and force and,
for the bond-based material, the damage Z, phi and the strain energy of every
node, for the state-based one the dilatation.  A quasi-static case solves one
load step.  A model goes on from where the pass before left it, as a program
does.  Setup (mesh, neighbor search, data layout, initial forces) is
prepare(): a program does it once per model.

The specimens are those of nlmech_amd.problems, of the sizes and options that
its workloads, tests and benchmark use: notched plates (horizon 3 h on
h = 1e-3 m, 4 h on h = 1e-4 m), blocks with pulled faces, ensembles of uneven
plates, clamped quasi-static plates.  Every specimen has a seeded mesh jitter
and, where it moves, a seeded initial velocity of 1e-3 m/s.
"""
import math

import numpy as np
import torch

from nlmech_amd import problems as pr
from nlmech_amd.capi import (NLM_PREC_FP32_FORCE, NLM_PREC_FP64,
                             NLM_PREC_FP64_EXACT, NLM_TIME_CENTRAL_DIFFERENCE,
                             NLM_TIME_VELOCITY_VERLET)
from nlmech_amd.engine import GpuFD

PRECISION = {"exact": NLM_PREC_FP64_EXACT, "fp64": NLM_PREC_FP64,
             "fp32": NLM_PREC_FP32_FORCE}
E, GC, RHO = 3.24e9, 500.0, 1200.0          # bond-based material
ES_K, ES_G, ES_SC = 2.16e9, 1.30e9, 1e-3    # state-based material
LAYERS = 3                                  # node rows of a loaded edge
LOAD = 1e8                                  # N/m^3, force-loaded edge


def plate(name, nx, ny, ratio, precision, steps, *, pull=0.5, jitter=1e-6,
          scheme="cd", influence=0, load="pull"):
    return dict(name=name, kind="plate", nx=nx, ny=ny, nz=1, ratio=ratio,
                precision=precision, steps=steps, pull=pull, jitter=jitter,
                scheme=scheme, influence=influence, load=load)


def block(name, kind, nx, ny, nz, precision, steps, *, pull):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, ratio=3,
                precision=precision, steps=steps, pull=pull, jitter=1e-6,
                scheme="cd", influence=0, load="pull")


def listed():
    return [
        # the 1e4-node plate at the default precision (the reference's own
        # arithmetic), 50 steps between outputs: launches and the read-back
        # count
        plate("plate 100x100 exact", 100, 100, 3, "exact", 50),
        # a fracture run at the default precision: fast pulls, bonds break
        # all the time
        plate("plate 400x397 exact breaking", 400, 397, 4, "exact", 200,
              pull=30.0),
        # velocity Verlet on an unstructured mesh (ragged rows), the linear
        # influence function, one edge loaded by a force
        plate("plate 333x217 fp64 verlet", 333, 217, 3, "fp64", 200,
              jitter=0.2, scheme="verlet", influence=1, load="force"),
        # a medium plate in FP64
        plate("plate 619x451 fp64", 619, 451, 4, "fp64", 300),
        # the 1e6-node plate in the FP32-force mode: the largest single run
        plate("plate 1000x1000 fp32", 1000, 1000, 4, "fp32", 600),
        # a parameter study: uneven notched plates packed into one model and
        # stepped from a captured graph
        dict(name="ensemble 16 plates fp32", kind="ensemble", count=16, lo=50,
             hi=300, ratio=3, precision="fp32", steps=200),
        # bond-based blocks
        block("block 41x37x45 fp64", "block", 41, 37, 45, "fp64", 100,
              pull=1.0),
        block("block 72x64x56 fp32", "block", 72, 64, 56, "fp32", 100,
              pull=0.5),
        # state-based blocks: the FP32-force mode at half a million nodes,
        # and the default precision with breaking bonds
        block("state block 80x80x80 fp32", "state_block", 80, 80, 80, "fp32",
              100, pull=0.3),
        block("state block 47x39x33 exact", "state_block", 47, 39, 33,
              "exact", 100, pull=1.0),
        # a state-based plate (plane stress)
        dict(block("state plate 301x257 fp64", "state_plate", 301, 257, 1,
                   "fp64", 200, pull=0.3)),
        # one load step of the quasi-static Newton solver
        dict(name="quasistatic 200x200", kind="quasistatic", nx=200, ny=200,
             nz=1, ratio=3, coarse=False),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["plate"] * 4 + ["block"] * 2 + ["state_block"] * 2 +
                      ["state_plate", "ensemble", "quasistatic"])
    prec = rng.choice(["exact", "fp64", "fp32"])
    if kind == "plate":
        ratio = rng.choice([3, 4])
        nx, ny = log(40, 700), log(40, 700)
        c = plate("", nx, ny, ratio, prec, log(10, 300),
                  jitter=rng.choice([1e-6, 1e-6, 0.2]),
                  scheme=rng.choice(["cd", "cd", "cd", "verlet"]),
                  influence=rng.choice([0, 0, 1]),
                  load=rng.choice(["pull", "pull", "force"]))
        # (broken-bond sets of the FP32-force mode depend on its rounding
        # once cracks run, so its specimens are pulled slowly)
        if prec != "fp32":
            c["pull"] = rng.choice([0.5, 30.0])
    elif kind in ("block", "state_block"):
        c = block("", kind, log(14, 70), log(14, 70), log(14, 70), prec,
                  log(10, 100), pull=0.3 if prec == "fp32" else 1.0)
    elif kind == "state_plate":
        c = block("", kind, log(40, 400), log(40, 400), 1, prec, log(10, 200),
                  pull=0.3)
    elif kind == "ensemble":
        lo = rng.randint(30, 100)
        c = dict(kind=kind, count=rng.randint(3, 20), lo=lo,
                 hi=lo + rng.randint(10, 150), ratio=3, precision=prec,
                 steps=2 * log(20, 100))
    else:
        n = rng.randint(40, 200)
        c = dict(kind=kind, nx=n, ny=n, nz=1, ratio=3,
                 coarse=rng.random() < 0.5)
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- specimens


def problem(c, seed):
    """The specimen of a case: nlmech_amd.problems.Problem."""
    kind = c["kind"]
    if kind == "ensemble":
        # (sides and notches belong to the case, the motion to the seed)
        p = pr.ensemble(count=c["count"], lo=c["lo"], hi=c["hi"],
                        ratio=c["ratio"], seed=3)
        return pr.with_(p, v0=velocity(p.n, 2, seed))
    if kind == "quasistatic":
        return pr.qs_plate(c["nx"], ratio=c["ratio"], pull=2e-6, seed=seed,
                           notch_len=0.1 * c["nx"] * 1e-3)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    dim = 2 if kind in ("plate", "state_plate") else 3
    if kind == "plate":
        h, dt = (1e-3, 1e-7) if c["ratio"] == 3 else (1e-4, 1e-8)
    else:
        h, dt = 6.25e-4, 5e-8
    if dim == 2:
        x, vol = pr.grid2d(nx, ny, h, c["jitter"], seed)
    else:
        x, vol = pr.grid3d(nx, ny, nz, h, c["jitter"], seed)
    # the loaded edge rows (2D: bottom and top, 3D: the z faces)
    axis, m = (1, ny) if dim == 2 else (2, nz)
    reach = max(nx, ny, nz) * h
    region = "rectangle" if dim == 2 else "cuboid"

    def rows(first, last):
        b = dict(x1=-h, x2=reach, y1=-h, y2=reach, z1=-h, z2=reach)
        key = "xyz"[axis]
        b[key + "1"], b[key + "2"] = (first - 0.5) * h, (last + 0.5) * h
        return b

    ubc, fbc = [], []
    ubc.append(pr.BC(region, [axis + 1], "linear", [-c["pull"]],
                     **rows(0, LAYERS - 1)))
    if c["load"] == "pull":
        ubc.append(pr.BC(region, [axis + 1], "linear", [c["pull"]],
                         **rows(m - LAYERS, m - 1)))
    else:
        fbc.append(pr.BC(region, [axis + 1], "constant", [LOAD],
                         **rows(m - LAYERS, m - 1)))
    cracks = []
    if kind == "plate":  # a notch of a fifth of the width at mid-height
        y = (ny // 2 - 0.5) * h
        cracks.append(pr.CrackSpec(1, (-0.5 * h, y),
                                   ((nx // 5 - 0.5) * h, y)))
    mat = (pr.rnp_material(dim=dim, E=E, Gc=GC, density=RHO,
                           inf_type=c["influence"],
                           inf_params=(1.0,) if c["influence"] == 0 else ())
           if kind in ("plate", "block") else
           pr.es_material(dim=dim, K=ES_K, G=ES_G, density=RHO, sc=ES_SC))
    return pr.Problem(name=kind, dim=dim, x=x, vol=vol, horizon=c["ratio"] * h,
                      h=h, dt=dt, nsteps=c["steps"], material=mat, ubc=ubc,
                      fbc=fbc, cracks=cracks, shape=(nx, ny, nz),
                      v0=velocity(x.shape[0], dim, seed))


def velocity(n, dim, seed):
    v = np.zeros((n, 3))
    v[:, :dim] = 1e-3 * np.random.default_rng(seed).standard_normal((n, dim))
    return v


def scheme_of(c):
    return (NLM_TIME_VELOCITY_VERLET if c.get("scheme") == "verlet"
            else NLM_TIME_CENTRAL_DIFFERENCE)


def prepare(case, seed):
    fd = GpuFD(problem(case, seed),
               precision=PRECISION[case.get("precision", "fp64")],
               scheme=scheme_of(case))
    if case["kind"] != "quasistatic":
        fd.init()
    return dict(case, fd=fd)


def run(state):
    fd, kind = state["fd"], state["kind"]
    if kind == "quasistatic":
        fd.qs_solve(1, dt=1.0, tol_rel=1e-8, lin_tol=1e-8,
                    precond=17 if state["coarse"] else 1)
        u, _, _ = fd.get_state()
        z, phi, energy = fd.postproc()
        return {"u": u, "Z": z, "phi": phi, "energy": energy}
    if kind == "ensemble":
        fd.step_graph(state["steps"], 50)
    else:
        fd.step(state["steps"])
    u, v, f = fd.get_state()
    out = {"u": u, "v": v, "f": f}
    if kind.startswith("state"):
        out["theta"] = fd.node_fields()[0]
    else:
        out["Z"], out["phi"], out["energy"] = fd.postproc()
    return out


# ------------------------------------------------------- compulsory work


def counts(c):
    """(nodes, directed bonds) of the unperturbed specimen."""
    if c["kind"] == "ensemble":
        side = 0.5 * (c["lo"] + c["hi"])
        shapes = [(side, side, 1)] * c["count"]
    else:
        shapes = [(c["nx"], c["ny"], c["nz"])]
    r = c["ratio"]
    n = bonds = 0
    for s in shapes:
        n += s[0] * s[1] * s[2]
        for a in range(-r, r + 1):
            for b in range(-r, r + 1):
                for d in range(-r, r + 1) if s[2] > 1 else (0,):
                    if 0 < a * a + b * b + d * d < r * r:
                        bonds += (max(0, s[0] - abs(a)) *
                                  max(0, s[1] - abs(b)) *
                                  max(0, s[2] - abs(d)))
    return n, bonds


def work(case):
    """Per force evaluation: positions, displacements, velocities, volumes,
    flags, row offsets read and the new displacements and velocities written
    once per node; a 4-byte column and a damage bit read once per bond.  An
    output: u, v, f and the damage or dilatation fields once per node."""
    n, bonds = counts(case)
    kind = case["kind"]
    if kind == "quasistatic":
        # about 5 sqrt(n) Krylov iterations, two products (a column and a
        # scalar per bond) and ten node vectors each
        its = 5.0 * math.sqrt(n)
        return {"bytes": its * (2 * 12.0 * bonds + 10 * 16.0 * n),
                "flops": its * (2 * 9.0 * bonds + 20.0 * n)}
    dim = 3 if kind in ("block", "state_block") else 2
    vec = 8.0 * dim
    node, bond, flop = 5 * vec + 13.0, 4.125, 16.0 + 8.0 * dim
    if kind.startswith("state"):
        node, bond, flop = node + 2 * vec + 40.0, 8.25, 2 * flop
    return {"bytes": case["steps"] * (node * n + bond * bonds) +
                     (3 * 24.0 + 16.0) * n,
            "flops": case["steps"] * (flop * bonds + 8.0 * dim * n)}


def tolerance(case):
    """About four times the largest error against exact().  FP64: the damage
    fields Z and phi are returned in FP32 (1.0e-7; u, v, f and the energy are
    within 5e-13, with the state-based extension's cancellation 3e-10).
    FP32-force: forces 2e-6.  Quasi-static: Z in FP32 at the solver's
    tolerance (1.2e-7)."""
    if case["kind"] == "quasistatic":
        return {"rel": 5e-7, "max": 1e-5}
    if case.get("precision") == "fp32":
        return {"rel": 8e-6, "max": 5e-4}
    return {"rel": 4e-7, "max": 4e-6}


# --------------------------------------------- the same in plain torch, FP64

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")


def greater(a, b):
    """The reference's relative-epsilon comparison a > b."""
    return (a - b) > 1e-5 * torch.maximum(a.abs(), b.abs())


class Rows:
    """Neighbor rows as an (n, W) table: candidate lattice offsets of every
    node's grid, masked by the neighbor predicate."""

    def __init__(self, p, grids, ratio, jitter):
        n, dim = p.n, p.dim
        self.x = torch.from_numpy(p.x).to(DEV)[:, :dim].contiguous()
        self.vol = torch.from_numpy(p.vol).to(DEV)
        reach = ratio + 3.0 * jitter
        k = int(math.ceil(reach))
        r = range(-k, k + 1)
        offs = [(a, b, d) for d in (r if dim == 3 else (0,)) for b in r
                for a in r if 0 < a * a + b * b + d * d <= reach * reach]
        self.nbr = torch.arange(n, device=DEV)[:, None].repeat(1, len(offs))
        ok = torch.zeros((n, len(offs)), dtype=torch.bool, device=DEV)
        for base, (nx, ny, nz) in grids:
            i = torch.arange(nx * ny * nz, device=DEV)
            ix, iy, iz = i % nx, (i // nx) % ny, i // (nx * ny)
            for w, (a, b, d) in enumerate(offs):
                inside = ((ix + a >= 0) & (ix + a < nx) & (iy + b >= 0) &
                          (iy + b < ny) & (iz + d >= 0) & (iz + d < nz))
                src = i[inside] + base
                self.nbr[src, w] = src + (a + nx * (b + ny * d))
                ok[src, w] = True
        dx = self.x[self.nbr] - self.x[:, None]
        r = dx.square().sum(-1).sqrt()
        eps = torch.tensor(p.horizon + 1e-10, dtype=torch.float64, device=DEV)
        self.ok = ok & greater(eps, r)
        used = self.ok.any(0)
        self.nbr, self.ok = self.nbr[:, used], self.ok[:, used]
        self.dx, self.r = dx[:, used], r[:, used]
        self.r[~self.ok] = 1.0
        # volume of the neighbor with the horizon-edge correction
        low = torch.tensor(p.horizon - 0.5 * p.h, dtype=torch.float64,
                           device=DEV)
        fac = torch.where(greater(self.r, low),
                          (p.horizon + 0.5 * p.h - self.r) / p.h, 1.0)
        self.volc = torch.where(self.ok, self.vol[self.nbr] * fac, 0.0)

    def diff(self, u):
        return u[self.nbr] - u[:, None]


def notch(rows, p, broken):
    """Bonds that cross a pre-crack."""
    for c in p.cracks:
        x = rows.x
        zero = torch.zeros((), dtype=torch.float64, device=DEV)
        rel = x - torch.tensor(c.pb, dtype=torch.float64, device=DEV)
        t = (c.pt[0] - c.pb[0], c.pt[1] - c.pb[1])
        if c.o == 1:
            lo, hi = zero + c.pb[0], zero + c.pt[0]
            out = greater(lo, x[:, 0]) | greater(x[:, 0], hi)
        else:
            out = greater(zero, rel[:, 0]) | greater(rel[:, 0], zero + t[0])
        left = ~greater(zero, 0.5 * (t[0] * rel[:, 1] - rel[:, 0] * t[1]))
        j = rows.nbr
        broken |= (~out[:, None] & ~out[j] & (left[:, None] != left[j]) &
                   rows.ok)


class BondBased:
    """RNP bonds: F = 4 C beta J S exp(-beta r S^2) / (pi eps^3 or 4 pi eps^4
    / 3) V_j e, broken once |S| exceeds sqrt(0.5 / beta) / sqrt(r)."""

    def __init__(self, rows, p, influence):
        self.rows = rows
        dim, eps = p.dim, p.horizon
        if influence == 0:
            a, b = 1.0, 0.0
        else:  # default linear influence function a (1 - r)
            a = 12.0 if dim == 2 else 20.0
            b = -a
        moment = a / (dim + 1) + b / (dim + 2)
        nu = 1.0 / 3.0
        lam = E * nu / ((1 + nu) * (1 - 2 * nu))
        if dim == 2:
            self.C = math.pi * GC / (4 * moment)
            self.beta = 4 * lam / (self.C * moment)
            norm = math.pi * eps ** 3
        else:
            self.C = 2 * GC / (3 * moment)
            self.beta = 5 * lam / (self.C * moment)
            norm = 4 * math.pi * eps ** 4 / 3
        r = rows.r
        self.infl = (a + b * r / eps) / norm
        self.crit = math.sqrt(0.5 / self.beta) / r.sqrt()
        # force per unit S exp(-beta r S^2), along dx / r
        self.k = 4 * self.C * self.beta * self.infl * rows.volc / r
        self.w = rows.dx / r.square()[..., None]
        self.broken = torch.zeros_like(rows.ok)
        notch(rows, p, self.broken)

    def stretch(self, u):
        return (self.rows.diff(u) * self.w).sum(-1)

    def force(self, u):
        s = self.stretch(u)
        self.broken |= greater(s.abs(), self.crit) & self.rows.ok
        g = self.k * s * torch.exp(-self.beta * self.rows.r * s * s)
        g[self.broken] = 0.0
        return (g[..., None] * self.rows.dx).sum(1)

    def fields(self, u):
        rows, s = self.rows, self.stretch(u)
        self.broken |= greater(s.abs(), self.crit) & rows.ok
        z = torch.where(rows.ok, s.abs() / self.crit, 0.0).amax(1)
        live = torch.where(self.broken, 0.0, rows.volc)
        phi = 1 - live.sum(1) / rows.volc.sum(1)
        e = 1 - torch.exp(-self.beta * rows.r * s * s)
        e[self.broken] = 1.0
        e = (self.C * self.infl * e * rows.volc).sum(1) * rows.vol
        return {"Z": z, "phi": phi, "energy": e}


class StateBased:
    """The linear state-based solid: dilatation, then the force of both
    directions of every bond; bonds break at the critical stretch."""

    def __init__(self, rows, p):
        self.rows, self.dim = rows, p.dim
        self.m = (rows.r.square() * rows.volc).sum(1)
        self.broken = torch.zeros_like(rows.ok)
        nu = (3 * ES_K - 2 * ES_G) / (2 * (3 * ES_K + ES_G))
        if p.dim == 2:  # plane stress
            self.f2 = (2 * nu - 1) / (nu - 1)
            kc = ES_K + ((nu + 1) / (2 * nu - 1)) ** 2 * ES_G / 9
            self.lead = 2 * self.f2 / self.m
            self.ad = 8 * ES_G / self.m
            self.c = (2 * self.f2 * 9 * kc / self.m -
                      (3 - 2 * self.f2) * self.ad)
        else:
            self.lead = 3 / self.m
            self.c = 9 * ES_K / self.m

    def force(self, u):
        rows = self.rows
        du = rows.diff(u)
        ly = (rows.dx + du).square().sum(-1).sqrt()
        ly[~rows.ok] = 1.0
        e = (du * (2 * rows.dx + du)).sum(-1) / (ly + rows.r)
        sc = torch.tensor(ES_SC, dtype=torch.float64, device=DEV)
        self.broken |= greater(e / rows.r, sc) & rows.ok
        live = torch.where(self.broken, 0.0, rows.volc)
        self.theta = self.lead * (rows.r * e * live).sum(1)
        j = rows.nbr
        if self.dim == 3:
            a = self.c * self.theta / 3
            t = (a[:, None] + a[j]) * rows.r
        else:
            a = self.theta * (self.c / 9 - self.ad / 3)
            t = ((a[:, None] + a[j]) * rows.r +
                 (self.ad[:, None] + self.ad[j]) * e)
        return ((t * live / ly)[..., None] * (rows.dx + du)).sum(1)

    def fields(self, u):
        return {"theta": self.theta}


def region(x, b, dim):
    keep = torch.ones(x.shape[0], dtype=torch.bool, device=DEV)
    for d in range(dim):
        key = "xyz"[d]
        keep &= ((x[:, d] >= getattr(b, key + "1")) &
                 (x[:, d] <= getattr(b, key + "2")))
    return keep


def padded(a, n):
    out = torch.zeros((n, 3), dtype=torch.float64, device=DEV)
    out[:, :a.shape[1]] = a
    return out


def exact(case, seed):
    p = problem(case, seed)
    if case["kind"] == "ensemble":
        grids = [(s["offset"], (s["side"], s["side"], 1))
                 for s in p.specimens]
    else:
        grids = [(0, (case["nx"], case["ny"], case["nz"]))]
    rows = Rows(p, grids, case["ratio"], case.get("jitter", 1e-6))
    bonds = (StateBased(rows, p) if case["kind"].startswith("state")
             else BondBased(rows, p, case.get("influence", 0)))
    n, dim, x = p.n, p.dim, rows.x
    rate = torch.zeros((n, dim), dtype=torch.float64, device=DEV)
    fixed = torch.zeros((n, dim), dtype=torch.bool, device=DEV)
    fext = torch.zeros((n, dim), dtype=torch.float64, device=DEV)
    for b in p.ubc:
        sel = region(x, b, dim)
        for d in b.dirs:
            fixed[sel, d - 1] = True
            rate[sel, d - 1] = (b.time_params[0] if b.time_fn == "linear"
                                else 0.0)
    for b in p.fbc:
        for d in b.dirs:
            fext[region(x, b, dim), d - 1] += b.time_params[0]
    if p.node_bc is not None:
        nodes, _, rates = p.node_bc
        at = torch.from_numpy(nodes).to(DEV)
        fixed[at, 1] = True
        rate[at, 1] = torch.from_numpy(rates[:, 1]).to(DEV)
    if case["kind"] == "quasistatic":
        u = newton(bonds, rows, fixed, rate)
        out = bonds.fields(u)
        out["u"] = padded(u, n)
        return {k: a.cpu() for k, a in out.items()}
    u = torch.zeros((n, dim), dtype=torch.float64, device=DEV)
    v = torch.from_numpy(p.v0).to(DEV)[:, :dim].contiguous()
    v = torch.where(fixed, rate, v)
    f, t, dt = fext + bonds.force(u), 0.0, p.dt
    for _ in range(case["steps"]):
        t += dt
        if case.get("scheme") == "verlet":
            v = v + 0.5 * dt / RHO * f
            u = torch.where(fixed, rate * t, u + dt * v)
            v = torch.where(fixed, rate, v)
            f = fext + bonds.force(u)
            v = torch.where(fixed, v, v + 0.5 * dt / RHO * f)
        else:
            v = torch.where(fixed, rate, v + dt / RHO * f)
            u = torch.where(fixed, rate * t, u + dt * v)
            f = fext + bonds.force(u)
    out = bonds.fields(u)
    out.update(u=padded(u, n), v=padded(v, n), f=padded(f, n))
    return {k: a.cpu() for k, a in out.items()}


def newton(bonds, rows, fixed, rate):
    """Equilibrium of one load step from rest: Newton with conjugate
    gradients on the tangent times the node volumes (symmetric)."""
    free = ~fixed
    vol = rows.vol[:, None]
    u = torch.zeros_like(rate)
    step = torch.where(fixed, rate, 0.0)
    for it in range(6):
        s = bonds.stretch(u)
        q = bonds.beta * rows.r * s * s
        k = bonds.k / rows.r.square() * torch.exp(-q) * (1 - 2 * q)
        k[bonds.broken] = 0.0

        def product(d):
            w = k * (rows.diff(d) * rows.dx).sum(-1)
            return -vol * (w[..., None] * rows.dx).sum(1)

        b = vol * bonds.force(u)
        if it == 0:  # the prescribed increment is Dirichlet data
            b = b - product(step)
        dg = vol * (k[..., None] * rows.dx.square()).sum(1)
        d = solve(lambda a: torch.where(free, product(a), 0.0),
                  torch.where(free, b, 0.0), dg)
        u = u + d + (step if it == 0 else 0.0)
        if it > 0 and float(d.norm()) <= 1e-13 * float(u.norm()):
            break
    return u


def solve(apply, b, dg):
    x = torch.zeros_like(b)
    r, z = b.clone(), b / dg
    p, rz = z.clone(), (b * z).sum()
    end = 1e-13 * float(b.norm())
    for k in range(6000):
        ap = apply(p)
        a = rz / (p * ap).sum()
        x += a * p
        r -= a * ap
        if k % 20 == 0 and float(r.norm()) <= end:
            break
        z = r / dg
        rz, old = (r * z).sum(), rz
        p = z + rz / old * p
    return x

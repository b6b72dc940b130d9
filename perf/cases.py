"""The work this framework is used for, as a set of measured cases.

Each case is one pass of a user's program through the public Python entry points (madpac_amd.lbm):
time stepping followed by the readout that the program asked for.  The sizes are those of this
repository's own configurations (README, bench.py, validate.py, tests) or generic ones around them.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and the solver object a program holds before the call
    run(state)           one pass; returns its outputs whole
    work(case)           the bytes and operations a pass cannot do without
    exact(case, seed)    the same outputs in 64-bit torch on the GPU, without the solver
"""
from __future__ import annotations

import math

import numpy as np
import torch

from madpac_amd import lbm

Q = 19
C = [(0, -1, -1), (-1, 0, -1), (0, 0, -1), (1, 0, -1), (0, 1, -1), (-1, -1, 0), (0, -1, 0), (1, -1, 0), (-1, 0, 0),
     (0, 0, 0), (1, 0, 0), (-1, 1, 0), (0, 1, 0), (1, 1, 0), (0, -1, 1), (-1, 0, 1), (0, 0, 1), (1, 0, 1), (0, 1, 1)]
W = [1 / 3 if c == (0, 0, 0) else (1 / 18 if sum(abs(v) for v in c) == 1 else 1 / 36) for c in C]
PRECISION = {"fp64": lbm.FP64, "fp32s": lbm.FP32_SHIFTED}
ESIZE = {"fp64": 8, "fp32s": 4}
FORCE = 1e-6           # Guo body force of the porous channel
LID, INLET = 0.05, 0.05
FLOPS_PER_UPDATE = 250  # moments, equilibrium and relaxation of one D3Q19 cell


# ---------------------------------------------------------------------------------------------
# cases
def _lattice(name, scene, size, precision, steps, layout="two_buffer", tune=False, monitors=0):
    nx, ny, nz = size
    c = {"kind": "lattice", "scene": scene, "nx": nx, "ny": ny, "nz": nz, "precision": precision, "steps": steps,
         "layout": layout, "tune": tune, "monitors": monitors}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: the smoke cavity, a handful of launch-bound steps and a readout
        _lattice("cavity_12_fp64", "cavity", (12, 12, 12), "fp64", 20),
        # the lid-driven cavity of the README (64^3, FP64, 1000 steps)
        _lattice("cavity_64_fp64", "cavity", (64, 64, 64), "fp64", 1000),
        # the reference's default channel in a box whose sides fit no tile, with a parabolic inlet and obstacles
        _lattice("channel_ragged_fp64", "channel", (131, 70, 53), "fp64", 300),
        # the porous channel of the benchmark, 256^3, in both precisions (tuned once, as bench.py does)
        _lattice("porous_256_fp64", "porous", (256, 256, 256), "fp64", 300, tune=True),
        _lattice("porous_256_fp32s", "porous", (256, 256, 256), "fp32s", 400, tune=True),
        # the Taylor-Green vortex with the energy and the moments monitored between stretches of steps
        _lattice("taylor_green_256_fp32s", "taylor_green", (256, 256, 256), "fp32s", 300, tune=True, monitors=6),
        # the in-place layout, for lattices whose second buffer does not fit
        _lattice("taylor_green_aa_fp64", "taylor_green", (256, 192, 160), "fp64", 200, layout="aa", tune=True),
        # uneven patches on tori, autotuned, replayed from a graph
        {"name": "patches_1024_fp32s", "kind": "patches", "count": 1024, "precision": "fp32s", "steps": 200},
        # the gradient of the pressure drop with respect to a porosity field (forward, recompute, reverse)
        {"name": "adjoint_duct_128_fp32s", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 128, "precision": "fp32s",
         "steps": 100, "snapshots": 12},
        # the reference's own iteration on its block layout
        {"name": "blocks_cavity_64", "kind": "blocks", "n": 64, "steps": 200},
        # one coarse time step's transfers between two grid levels: overlap search, prolongation, restriction
        {"name": "levels_512", "kind": "levels", "coarse": 512},
        # the MD coupling loop: new MD data, a few steps, export of the coupled cells
        {"name": "coupling_96_fp64", "kind": "coupling", "nx": 96, "ny": 96, "nz": 96, "box": 24, "exchanges": 20,
         "steps": 10},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lattice"] * 7 + ["patches", "patches", "adjoint", "blocks", "levels", "coupling"])
    precision = rng.choice(["fp64", "fp32s"])
    if kind == "lattice":
        scene = rng.choice(["cavity", "channel", "porous", "taylor_green"])
        lo = 24 if scene == "porous" else 12
        while True:
            e = _size(rng, lo, 256)
            nx, ny, nz = (max(10, int(round(e * rng.uniform(0.7, 1.3)))) for _ in range(3))
            if rng.random() < 0.4:  # boxes of whole 64-cell rows are common
                nx = max(64, 64 * round(nx / 64))
            if nx * ny * nz <= 256 ** 3:
                break
        cells = nx * ny * nz
        steps = rng.randint(20, max(21, int(min(1000, 6e9 / cells))))
        layout = rng.choice(["two_buffer", "two_buffer", "two_buffer", "aa"])
        return _lattice(None, scene, (nx, ny, nz), precision, min(steps, 300), layout, cells > 1 << 20,
                        rng.choice([0, 0, 3]))
    if kind == "patches":
        return {"kind": "patches", "count": _size(rng, 16, 1024), "precision": precision, "steps": rng.randint(20, 200)}
    if kind == "adjoint":
        nx, ny, nz = (rng.randint(20, 128) for _ in range(3))
        return {"kind": "adjoint", "nx": nx, "ny": ny, "nz": nz, "precision": precision, "steps": rng.randint(20, 90),
                "snapshots": rng.randint(4, 23)}
    if kind == "blocks":
        return {"kind": "blocks", "n": _size(rng, 12, 128), "steps": rng.randint(5, 100)}
    if kind == "levels":
        return {"kind": "levels", "coarse": _size(rng, 8, 512)}
    nx, ny, nz = (rng.randint(32, 128) for _ in range(3))
    return {"kind": "coupling", "nx": nx, "ny": ny, "nz": nz, "box": rng.randint(8, 28),
            "exchanges": rng.randint(5, 20), "steps": rng.randint(1, 10)}


# ---------------------------------------------------------------------------------------------
# inputs
def _spheres(nx, ny, nz, fraction, rmin, rmax, rng):
    """Bool (nz, ny, nx): spheres at random places until `fraction` of the box is solid (wrapping)."""
    solid = np.zeros((nz, ny, nx), bool)
    rmax = max(1, min(rmax, (min(nx, ny, nz) - 1) // 2))
    rmin = min(rmin, rmax)
    target, count = int(fraction * solid.size), 0
    while count < target:
        r = int(rng.integers(rmin, rmax + 1))
        o = np.arange(-r, r + 1)
        ball = o[:, None, None] ** 2 + o[None, :, None] ** 2 + o[None, None, :] ** 2 <= r * r
        at = [(int(rng.integers(0, n)) + o) % n for n in (nz, ny, nx)]
        sub = solid[np.ix_(*at)]
        solid[np.ix_(*at)] = sub | ball
        count += int((ball & ~sub).sum())
    return solid


def _waves(nx, ny, nz, rng, modes=3):
    """Smooth random field in [-1, 1] on the GPU, (nz, ny, nx) in FP64."""
    def axis(n, k, phase):
        return torch.cos(2 * math.pi * k * torch.arange(n, dtype=torch.float64, device="cuda") / n + phase)
    out = torch.zeros(nz, ny, nx, dtype=torch.float64, device="cuda")
    for _ in range(modes):
        k, ph = rng.integers(1, 4, 3), rng.uniform(0, 2 * math.pi, 3)
        out += (axis(nz, k[2], ph[2])[:, None, None] * axis(ny, k[1], ph[1])[None, :, None]
                * axis(nx, k[0], ph[0])[None, None, :])
    return out / modes


def _inputs(case, seed):
    """Geometry and initial fields of the lattice kinds: solid (numpy bool), rho and u (torch, GPU)."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    scene = case.get("scene", case["kind"])
    solid = np.zeros((nz, ny, nx), bool)
    amplitude = 0.01
    if scene == "porous":
        solid = _spheres(nx, ny, nz, 0.2, 4, 12, rng)
        amplitude = 0.002
    elif scene == "channel":
        inner = _spheres(nx, ny, nz, 0.03, 2, 6, rng)
        solid[:, :, nx // 4:nx // 2] = inner[:, :, nx // 4:nx // 2]
    elif scene == "adjoint":
        solid[0] = solid[-1] = True
        solid[:, 0] = solid[:, -1] = True
    elif scene == "taylor_green":
        amplitude = 0.04
    rho = 1.0 + 0.1 * amplitude * _waves(nx, ny, nz, rng)
    u = torch.stack([amplitude * _waves(nx, ny, nz, rng) for _ in range(3)], -1)
    return solid, rho, u


def _patch_inputs(case, seed):
    """The uneven-patch workload: edges 8, 16, 24, 32, patches of equal edge joined into 2 x 2 x 2
    tori (the rest of an edge class into one ring); the edges follow from the count, the relaxation
    times and velocities from the seed.  Returns (table, tori, u); a torus is (dims, n, first patch, taus)."""
    rng = np.random.default_rng(seed)
    edges = np.random.default_rng(case["count"]).choice(np.array([8, 16, 24, 32]), size=case["count"])
    table, tori = [], []
    for n in (8, 16, 24, 32):
        left = int((edges == n).sum())
        while left:
            size = 8 if left >= 8 else left
            a, b, c = (2, 2, 2) if size == 8 else (size, 1, 1)
            first = len(table)
            taus = rng.uniform(0.55, 1.5, size)
            for p in range(size):
                i, j, k = p % a, (p // a) % b, p // (a * b)
                nbr = [first + (i + d[0]) % a + a * ((j + d[1]) % b + b * ((k + d[2]) % c)) for d in C]
                table.append((n, float(taus[p]), nbr))
            tori.append(((a, b, c), n, first, taus))
            left -= size
    cells = sum(t[0] ** 3 for t in table)
    u = 0.01 * np.random.default_rng(seed + 1).standard_normal((cells, 3), dtype=np.float32).astype(np.float64)
    return table, tori, u


def _block_grid(n):
    """The n^3 cavity on 6^3 blocks: slot s of block b holds cell 6 b + s - 3 (x fastest)."""
    nb = n // 6 + 1 + (1 if n % 6 else 0)
    b, s = np.arange(nb ** 3), np.arange(216)
    xyz = [6 * v[:, None] + w[None, :] - 3 for v, w in
           ((b % nb, s % 6), ((b // nb) % nb, (s // 6) % 6), (b // nb ** 2, s // 36))]
    inner = np.logical_and.reduce([(v >= 0) & (v < n) for v in xyz])
    index = np.where(inner, xyz[0] + n * (xyz[1] + n * xyz[2]), 0)
    c0 = np.arange(nb - 1)
    cz, cy, cx = np.meshgrid(c0, c0, c0, indexing="ij")
    base = (cx + nb * (cy + nb * cz)).reshape(-1)
    cells = np.stack([base + (v & 1) + nb * ((v >> 1) & 1) + nb * nb * (v >> 2) for v in range(8)], 1).astype(np.int64)
    blk, cell = np.nonzero(inner & (xyz[2] == n - 1))
    links = np.zeros((len(blk), 5), lbm.BlockStore.LINK_DTYPE)
    links["block"], links["cell"] = blk[:, None], cell[:, None]
    links["q_in"], links["type"] = np.array([18 - q for q in range(14, 19)]), lbm.BOUNDARY_MOVING_WALL
    links["u"], links["rho"] = (LID, 0.0, 0.0), 1.0
    return nb ** 3, inner, index, cells, links.reshape(-1)


def _block_fields(case, seed):
    n = case["n"]
    rng = np.random.default_rng(seed)
    rho = 1.0 + 0.001 * _waves(n, n, n, rng)
    u = torch.stack([0.01 * _waves(n, n, n, rng) for _ in range(3)], -1)
    return _equilibrium(rho, [u[..., d] for d in range(3)])


def _to_blocks(values, inner, index, fill):
    """(cells, k) box values -> (blocks, 216 * k) with `fill` outside the box."""
    v = values.cpu().numpy()
    out = np.where(inner[..., None], v[index], np.asarray(fill))
    return np.ascontiguousarray(out.reshape(len(inner), -1))


def _level_inputs(case, seed):
    nc = case["coarse"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.tensor(W, dtype=torch.float64, device="cuda").repeat(216)
    pdf = w * (1.0 + 0.05 * torch.randn(9 * nc, 216 * Q, dtype=torch.float64, device="cuda", generator=g))
    octant = np.random.default_rng(seed).integers(0, 2, (nc, 3))
    links = []
    for cb in range(nc):
        for k in range(8):
            pos = tuple(int(2 * octant[cb, d] + ((k >> d) & 1)) for d in range(3))
            links.append((cb, nc + 8 * cb + k, pos, k % 3 == 0))  # every third fine vertex is new
    return pdf, links


def _coupled_cells(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    e = [min(case["box"], n) for n in (nx, ny, nz)]
    lo = [(n - m) // 2 for n, m in zip((nx, ny, nz), e)]
    z, y, x = np.meshgrid(*[np.arange(l, l + m) for l, m in zip(lo[::-1], e[::-1])], indexing="ij")
    return (x + nx * (y + ny * z)).reshape(-1).astype(np.int64)


def _md_velocity(case, seed):
    n = len(_coupled_cells(case))
    return 0.01 + 0.002 * np.random.default_rng(seed + 2).standard_normal((case["exchanges"], n, 3))


def _porosity(case, seed):
    rng = np.random.default_rng(seed + 3)
    return 0.5 + 0.45 * _waves(case["nx"], case["ny"], case["nz"], rng, 6)


def _open(case, seed):
    """The lattice of a lattice, coupling or adjoint case with its geometry, and the initial fields."""
    scene = case.get("scene", case["kind"])
    solid, rho, u = _inputs(case, seed)
    periodic = {"porous": (True,) * 3, "taylor_green": (True,) * 3, "adjoint": (True, False, False)}.get(scene, (False,) * 3)
    force = {"porous": (FORCE, 0.0, 0.0), "adjoint": (1e-5, 0.0, 0.0)}.get(scene, (0.0,) * 3)
    tau = 0.52 if scene == "taylor_green" else 0.6
    layout = lbm.LAYOUT_AA if case.get("layout") == "aa" else lbm.LAYOUT_TWO_BUFFER
    lat = lbm.Lattice(case["nx"], case["ny"], case["nz"], tau, precision=PRECISION[case.get("precision", "fp64")],
                      periodic=periodic, force=force, layout=layout)
    lat.set_flags(~solid)
    if scene in ("cavity", "coupling"):
        lat.set_cavity_lid(LID)
    elif scene == "channel":
        lat.set_channel(INLET, parabolic=True)
    return lat, rho.cpu().numpy(), u.cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        lat, rho, u = _open(case, seed)
        lat.init_equilibrium(rho, u)
        if case["tune"]:
            lat.tune(10)
        return {"case": case, "lat": lat}
    if kind == "patches":
        table, _, u = _patch_inputs(case, seed)
        ps = lbm.PatchSet(table, precision=PRECISION[case["precision"]])
        ps.init(u=u)
        ps.autotune()
        return {"case": case, "ps": ps}
    if kind == "adjoint":
        lat, rho, u = _open(case, seed)
        lat.set_porosity(_porosity(case, seed).cpu().numpy())
        lat.init_equilibrium(rho, u)
        return {"case": case, "lat": lat}
    if kind == "blocks":
        nblocks, inner, index, cells, links = _block_grid(case["n"])
        f = _block_fields(case, seed).reshape(Q, -1).T.contiguous()
        bs = lbm.BlockStore(nblocks)
        bs.set(0, pdf=_to_blocks(f, inner, index, W), density=np.ones((nblocks, 216)))
        bs.set_inner(0, inner)
        return {"case": case, "bs": bs, "blocks": np.arange(nblocks), "cells": cells, "links": links}
    if kind == "levels":
        pdf, links = _level_inputs(case, seed)
        bs = lbm.BlockStore(9 * case["coarse"])
        bs.set(0, pdf=pdf.cpu().numpy())
        return {"case": case, "bs": bs, "links": links}
    lat, rho, u = _open(case, seed)
    lat.init_equilibrium(rho, u)
    lat.set_coupling_cells(_coupled_cells(case))
    return {"case": case, "lat": lat, "md": _md_velocity(case, seed)}


# ---------------------------------------------------------------------------------------------
# one pass
def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "lattice":
        lat, steps, out = state["lat"], case["steps"], {}
        m = case["monitors"]
        for k in range(m):
            lat.step(steps // m)
            out["energy%d" % k] = lat.kinetic_energy()
            out["moments%d" % k] = lat.moments()
        lat.step(steps - m * (steps // m) if m else steps)
        if case["scene"] == "porous":
            out["drop"] = lat.pressure_drop(0, case["nx"] // 2)
        out["rho"], out["u"] = lat.fields()
        return out
    if kind == "patches":
        ps = state["ps"]
        ps.step(case["steps"], graph=True)
        rho, u = ps.fields()
        return {"rho": rho, "u": u}
    if kind == "adjoint":
        J, grad, _ = state["lat"].adjoint_pressure_drop(case["steps"], case["snapshots"], case["nx"] // 4,
                                                        3 * case["nx"] // 4)
        return {"J": J, "grad": grad}
    if kind == "blocks":
        bs = state["bs"]
        bs.iterate(state["blocks"], state["cells"], 0.6, state["links"], case["steps"])
        return dict(zip(("pdf", "rho", "u"), bs.get()))
    if kind == "levels":
        bs, links = state["bs"], state["links"]
        overlap = bs.find_overlap(links)
        bs.prolongate(links)
        bs.restrict(links)
        return {"overlap": overlap, "pdf": bs.get()[0]}
    lat, out = state["lat"], {}
    for k in range(case["exchanges"]):
        lat.set_coupling_data(lbm.COUPLE_DIRICHLET, state["md"][k], dt=1.0)
        lat.step(case["steps"])
        out["rho%d" % k], out["u%d" % k] = lat.get_coupling_data()
    return out


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without: the state read and written once, the outputs written once, and the
# operations of every cell update
def work(case):
    kind, e = case["kind"], ESIZE[case.get("precision", "fp64")]
    if kind in ("lattice", "coupling", "adjoint"):
        cells = case["nx"] * case["ny"] * case["nz"]
        fluid = 0.8 * cells if case.get("scene") == "porous" else cells
        if kind == "lattice":
            return {"bytes": fluid * 2 * Q * e + 32 * cells, "flops": fluid * FLOPS_PER_UPDATE * case["steps"]}
        if kind == "adjoint":  # a forward and a reverse update per step
            return {"bytes": cells * (2 * Q * e + e + 8), "flops": 3 * cells * FLOPS_PER_UPDATE * case["steps"]}
        m = len(_coupled_cells(case))
        return {"bytes": cells * 2 * Q * 8 + case["exchanges"] * m * 7 * 8,
                "flops": cells * FLOPS_PER_UPDATE * case["steps"] * case["exchanges"]}
    if kind == "patches":
        edges = np.random.default_rng(case["count"]).choice(np.array([8, 16, 24, 32]), size=case["count"])
        cells = int((edges ** 3).sum())
        return {"bytes": cells * (2 * Q * e + 32), "flops": cells * FLOPS_PER_UPDATE * case["steps"]}
    if kind == "blocks":
        cells = case["n"] ** 3
        return {"bytes": cells * (2 * Q + 8) * 8, "flops": cells * FLOPS_PER_UPDATE * case["steps"]}
    fine = 8 * case["coarse"]
    return {"bytes": (case["coarse"] + fine) * 2 * 216 * Q * 8, "flops": fine * 216 * Q}


# ---------------------------------------------------------------------------------------------
# 64-bit values of the same outputs (plain torch on the GPU, pull form of the lattice update)
def _equilibrium(rho, v):
    uu = v[0] * v[0] + v[1] * v[1] + v[2] * v[2]
    out = []
    for q in range(Q):
        cu = sum(c * a for c, a in zip(C[q], v) if c)
        out.append(W[q] * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * uu))
    return torch.stack(out)


class _Exact:
    """D3Q19 BGK on a box (any leading batch axes of f[q] before z, y, x)."""

    def __init__(self, shape, tau, solid=None, periodic=(True,) * 3, force=(0.0,) * 3, lid=None, inlet=None):
        # as the solver derives it: nu = (tau - 1/2) / 3, tau_eff = 3 nu + 1/2
        self.tau, self.periodic, self.force, self.lid, self.inlet = tau, periodic, force, lid, inlet
        nz, ny, nx = shape
        closed = torch.zeros(shape, dtype=torch.bool, device="cuda") if solid is None else torch.as_tensor(solid, device="cuda")
        self.fluid = ~closed
        self.open_box = solid is None and all(periodic)
        self.wall = []
        for q in range(Q):  # whether x - c_q is no fluid cell
            c = C[q]
            b = torch.roll(closed, (c[2], c[1], c[0]), (0, 1, 2)).clone()
            for d, (axis, p) in enumerate(((2, periodic[0]), (1, periodic[1]), (0, periodic[2]))):
                if c[d] and not p:
                    b.narrow(axis, 0 if c[d] > 0 else shape[axis] - 1, 1).fill_(True)
            self.wall.append(b)
        if inlet is not None:
            a = [(torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) for n in (ny, nz)]
            self.profile = (inlet * (6.0 / ny ** 2 * a[0] * (ny - a[0]))[None, :] * (6.0 / nz ** 2 * a[1] * (nz - a[1]))[:, None])

    def moments(self, f):
        rho = f.sum(0)
        v = [sum(C[q][d] * f[q] for q in range(Q) if C[q][d]) / rho for d in range(3)]
        return rho, v

    def collide(self, f, alpha=None, coupled=None):
        rho, v = self.moments(f)
        g = self.force
        forced = any(g)
        if forced:
            v = [a + 0.5 * b for a, b in zip(v, g)]
        u = v
        if alpha is not None:
            v = [(1.0 - alpha) * a for a in v]
        if coupled is not None:
            cells, um = coupled
            gd = []
            for d in range(3):
                full = torch.zeros_like(rho).reshape(-1)
                full[cells] = um[:, d] - v[d].reshape(-1)[cells]
                gd.append(full.reshape(rho.shape))
            v = [a + 0.5 * b for a, b in zip(v, gd)]
        omega = 1.0 / self.tau
        uu = v[0] * v[0] + v[1] * v[1] + v[2] * v[2]
        out = []
        for q in range(Q):
            cu = sum(c * a for c, a in zip(C[q], v) if c)
            feq = W[q] * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * uu)
            s = f[q] - omega * (f[q] - feq)
            if forced:
                cg = sum(c * a for c, a in zip(C[q], g))
                ug = sum(a * b for a, b in zip(v, g))
                s = s + (1.0 - 0.5 * omega) * W[q] * rho * (3.0 * (cg - ug) + 9.0 * cu * cg)
            if coupled is not None:  # the coupling's forcing term, with (c.u)^2
                cg = sum(c * a for c, a in zip(C[q], gd))
                cmg = cg - sum(a * b for a, b in zip(v, gd))
                s = s + (1.0 - 0.5 * omega) * W[q] * rho * (3.0 * cmg + 9.0 * cu * cu * cg)
            out.append(s)
        return out, rho, u

    def step(self, f, alpha=None, coupled=None):
        s, rho, u = self.collide(f, alpha, coupled)
        new = []
        for q in range(Q):
            c, o = C[q], Q - 1 - q
            moved = torch.roll(s[q], (c[2], c[1], c[0]), (-3, -2, -1)) if any(c) else s[q]
            if not self.open_box and any(c):
                back = s[o]  # the outgoing population o = 18 - q of this cell
                co = C[o]
                if self.lid is not None and co[2] > 0 and co[0]:
                    back = back.clone()
                    back[-1] -= 6.0 * W[o] * rho[-1] * self.lid * co[0]
                if self.inlet is not None and co[0]:
                    back = self._open_faces(back, o, rho, u)
                moved = torch.where(self.wall[q], back, moved)
            new.append(moved)
        return torch.stack(new)

    def _open_faces(self, back, o, rho, u):
        """The channel's x faces for outgoing link o; a link that also leaves through y or z is a wall."""
        back, co = back.clone(), C[o]
        nz, ny, nx = back.shape
        y = slice(max(0, -co[1]), ny - max(0, co[1]))
        z = slice(max(0, -co[2]), nz - max(0, co[2]))
        if co[0] < 0:
            v = self.profile[z, y]
            cu = -co[0] * v  # the incoming direction
            back[z, y, 0] = W[o] * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * v * v)
        else:
            w = [a[z, y, -1] for a in u]
            cu = sum(c * a for c, a in zip(co, w) if c)
            uu = sum(a * a for a in w)
            back[z, y, -1] = -back[z, y, -1] + 2.0 * W[o] * (1.0 + 4.5 * cu * cu - 1.5 * uu)
        return back

    def fields(self, f):
        rho, v = self.moments(f)
        zero = torch.zeros_like(rho)
        return (torch.where(self.fluid, rho, zero).reshape(-1),
                torch.stack([torch.where(self.fluid, a, zero) for a in v], -1).reshape(-1, 3))


def _exact_box(case, seed):
    scene = case.get("scene", case["kind"])
    solid, rho, u = _inputs(case, seed)
    f = _equilibrium(rho, [u[..., d] for d in range(3)])
    shape = (case["nz"], case["ny"], case["nx"])
    if scene == "porous":
        return _Exact(shape, 0.6, solid, force=(FORCE, 0.0, 0.0)), f
    if scene == "taylor_green":
        return _Exact(shape, 0.52), f
    if scene == "adjoint":
        return _Exact(shape, 0.6, solid, (True, False, False), (1e-5, 0.0, 0.0)), f
    if scene == "channel":
        return _Exact(shape, 0.6, solid, (False,) * 3, inlet=INLET), f
    return _Exact(shape, 0.6, solid, (False,) * 3, lid=LID), f


def _drop(E, f, xin, xout):
    d = f.sum(0) - 1.0
    mean = [torch.where(E.fluid[..., x], d[..., x], torch.zeros_like(d[..., x])).sum() / E.fluid[..., x].sum()
            for x in (xin, xout)]
    return (mean[0] - mean[1]) / 3.0


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        E, f = _exact_box(case, seed)
        steps, m, out = case["steps"], case["monitors"], {}
        todo = [steps // m] * m + [steps - m * (steps // m)] if m else [steps]
        for k, n in enumerate(todo):
            for _ in range(n):
                f = E.step(f)
            if k < m:
                rho, u = E.fields(f)
                j = rho[:, None] * u
                safe = torch.where(rho > 0, rho, torch.ones_like(rho))
                out["energy%d" % k] = float((j.square().sum(1) / (2.0 * safe)).sum())
                out["moments%d" % k] = torch.cat([rho.sum()[None], j.sum(0)])
        if case["scene"] == "porous":
            out["drop"] = float(_drop(E, f, 0, case["nx"] // 2))
        out["rho"], out["u"] = E.fields(f)
        return out
    if kind == "patches":
        table, tori, u0 = _patch_inputs(case, seed)
        u0 = torch.from_numpy(u0).cuda()
        start = np.concatenate([[0], np.cumsum([t[0] ** 3 for t in table])])
        rho_out, u_out = torch.empty(len(u0), dtype=torch.float64, device="cuda"), torch.empty_like(u0)
        for key in sorted({(d, n) for d, n, _, _ in tori}):
            (a, b, c), n = key
            same = [t for t in tori if (t[0], t[1]) == key]
            size = a * b * c * n ** 3
            at = torch.cat([torch.arange(int(start[t[2]]), int(start[t[2]]) + size, device="cuda") for t in same])

            def to_box(v):  # (tori, patches z y x, n n n, k) -> k x (tori, z, y, x)
                v = v.reshape(len(same), c, b, a, n, n, n, -1).permute(7, 0, 1, 4, 2, 5, 3, 6)
                return v.reshape(v.shape[0], len(same), c * n, b * n, a * n)

            def from_box(v):
                v = v.reshape(-1, len(same), c, n, b, n, a, n).permute(1, 2, 4, 6, 3, 5, 7, 0)
                return v.reshape(len(same) * size, -1)

            tau = torch.tensor(np.stack([t[3] for t in same]), device="cuda")
            tau = to_box(tau[:, :, None].expand(-1, -1, n ** 3).reshape(-1, 1))[0]
            E = _Exact((c * n, b * n, a * n), tau)
            v = to_box(u0[at])
            f = _equilibrium(torch.ones_like(v[0]), list(v))
            for _ in range(case["steps"]):
                f = E.step(f)
            rho, v = E.moments(f)
            rho_out[at] = from_box(rho[None])[:, 0]
            u_out[at] = from_box(torch.stack(v))
        return {"rho": rho_out, "u": u_out}
    if kind == "adjoint":
        E, f = _exact_box(case, seed)
        alpha = _porosity(case, seed)
        states = []
        for _ in range(case["steps"]):
            states.append(f)
            f = E.step(f, alpha)
        xin, xout = case["nx"] // 4, 3 * case["nx"] // 4
        grad = torch.zeros_like(alpha)
        with torch.enable_grad():
            f = f.detach().requires_grad_(True)
            J = _drop(E, f, xin, xout)
            lam, = torch.autograd.grad(J, f)
            while states:
                s = states.pop().detach().requires_grad_(True)
                al = alpha.detach().requires_grad_(True)
                lam, ga = torch.autograd.grad(E.step(s, al), (s, al), lam)
                grad += ga
        grad = torch.where(E.fluid, grad, torch.zeros_like(grad))
        return {"J": float(J), "grad": grad.reshape(-1)}
    if kind == "blocks":
        nblocks, inner, index, _, _ = _block_grid(case["n"])
        E = _Exact((case["n"],) * 3, 0.6, np.zeros((case["n"],) * 3, bool), (False,) * 3, lid=LID)
        f = _block_fields(case, seed)
        for _ in range(case["steps"]):
            last, f = f, E.step(f)
        rho, u = E.fields(last)  # the blocks hold the values computed before the last collision
        return {"pdf": _to_blocks(f.reshape(Q, -1).T, inner, index, W), "rho": _to_blocks(rho[:, None], inner, index, 1.0),
                "u": _to_blocks(u, inner, index, 0.0)}
    if kind == "levels":
        pdf, links = _level_inputs(case, seed)
        pdf = pdf.reshape(-1, 6, 6, 6, Q)  # block, z, y, x, q
        sub = torch.tensor([1, 2, 0, 1])
        lk = torch.tensor([[l[0], l[1], *l[2], int(l[3])] for l in links])
        lo = (2 * sub[lk[:, 2:5]]).cuda()
        cb, fb, new = lk[:, 0].cuda(), lk[:, 1].cuda(), lk[:, 5].cuda() == 1
        fine = torch.arange(6, device="cuda") // 3
        x, y, z = (lo[:, d, None] + fine for d in range(3))
        taken = pdf[cb[:, None, None, None], z[:, :, None, None], y[:, None, :, None], x[:, None, None, :]]
        pdf[fb] = torch.where(new[:, None, None, None, None], taken, pdf[fb])
        mean = pdf[fb].reshape(-1, 2, 3, 2, 3, 2, 3, Q).mean((2, 4, 6))
        half = torch.arange(2, device="cuda")
        x, y, z = (lo[:, d, None] + half for d in range(3))
        pdf[cb[:, None, None, None], z[:, :, None, None], y[:, None, :, None], x[:, None, None, :]] = mean
        return {"overlap": None, "pdf": pdf.reshape(-1, 216 * Q)}
    E, f = _exact_box(case, seed)
    cells = torch.from_numpy(_coupled_cells(case)).cuda()
    md, out = torch.from_numpy(_md_velocity(case, seed)).cuda(), {}
    for k in range(case["exchanges"]):
        for _ in range(case["steps"]):
            f = E.step(f, coupled=(cells, md[k]))
        rho, v = E.moments(f)
        u = torch.stack([a.reshape(-1)[cells] for a in v], -1)
        out["rho%d" % k] = rho.reshape(-1)[cells]
        out["u%d" % k] = u + 0.5 * (md[k] - u)  # the export passes through the coupling's update
    return out

"""Timed workloads of the engine, through its public entry points.

Each case is one thing a program does with the library: a time loop of the
README program (dense, sparse, corrected and 2D grids), a loop written as
separate update / P2G / G2P calls, a @G2P2G loop, a batch of scenes, a
checkpointed rollout with its pullback, and the block partition.  Sizes are
those of the scenes in tesserae_hip.scenes and of bench.py, and sizes between
them.  ``exact`` restates the same pass in plain Float64 torch.

A case names its scene, the mesh cells per unit length ("cells"; for the rod
the cells per radius), the basis, the scalar type, the storage layout, and how
many steps one call of the path takes.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tesserae.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tesserae_hip as th  # noqa: E402

DEV = "cuda"
F32, F64 = torch.float32, torch.float64


def _dtype(case):
    return F32 if case["dtype"] == "f32" else F64


def _basis(name):
    k = {"linear": lambda: th.BSpline(th.Linear()), "quadratic": lambda: th.BSpline(th.Quadratic()),
         "cubic": lambda: th.BSpline(th.Cubic()), "ugimp": th.uGIMP}
    if name.startswith("kc_"):
        return th.KernelCorrection(k[name[3:]]())
    if name.startswith("wls_"):
        return th.WLS(k[name[4:]]())
    return k[name]()


def listed():
    return [
        # the README example: two 2D disks of 10,048 particles, Float64; the smallest program, bound by launches
        {"name": "disks_2d_f64", "path": "steps", "scene": "disks", "cells": 100, "basis": "quadratic",
         "dtype": "f64", "layout": "julia", "steps": 50, "reorder": 0.0, "speed": 0.1},
        # the headline: 13,434,880 particles of an elastic block, Float32, the loop's reorder check on
        {"name": "drop_3d_f32", "path": "steps", "scene": "drop", "cells": 256, "basis": "quadratic",
         "dtype": "f32", "layout": "julia", "steps": 10, "reorder": 0.85, "speed": 0.0},
        # the same block at 1/8 of the particles while it falls fast (particles change cells every step),
        # stepped with a call per output frame of a few steps
        {"name": "fall_3d_f32", "path": "steps", "scene": "drop", "cells": 128, "basis": "quadratic",
         "dtype": "f32", "layout": "julia", "steps": 5, "reorder": 0.85, "speed": 2.5},
        # the Taylor-impact rod of the reference's GPU example, Float64, kernel correction at the floor
        {"name": "rod_kc_f64", "path": "steps", "scene": "rod", "cells": 12, "basis": "kc_quadratic",
         "dtype": "f64", "layout": "julia", "steps": 5, "reorder": 0.85, "speed": 227.0},
        # the sparse-grid sphere at half its full resolution (15 M particles), cubic
        {"name": "sphere_cubic_f32", "path": "steps", "scene": "sphere", "cells": 256, "basis": "cubic",
         "dtype": "f32", "layout": "julia", "steps": 3, "reorder": 0.85, "speed": 0.5},
        # the same sphere at a quarter (1.9 M particles), uGIMP
        {"name": "sphere_ugimp_f32", "path": "steps", "scene": "sphere", "cells": 128, "basis": "ugimp",
         "dtype": "f32", "layout": "julia", "steps": 4, "reorder": 0.85, "speed": 0.5},
        # a loop body written as separate calls with stored weights, the reference's default form:
        # update!(weights), @P2G, @G2P; 2D, Float64
        {"name": "stored_2d_f64", "path": "calls", "scene": "box", "cells": 256, "basis": "quadratic",
         "dtype": "f64", "layout": "julia", "ppc": 4, "stored": True, "speed": 0.3},
        # separate @P2G and @G2P calls with deferred weights, 3D, Float32, particles in generation order
        {"name": "calls_3d_f32", "path": "calls", "scene": "drop", "cells": 128, "basis": "quadratic",
         "dtype": "f32", "layout": "julia", "stored": False, "speed": 1.0},
        # a @G2P2G loop on the block at 1/8 of the particles
        {"name": "g2p2g_3d_f32", "path": "g2p2g", "scene": "drop", "cells": 128, "basis": "quadratic",
         "dtype": "f32", "layout": "julia", "steps": 5, "reorder": 0.85, "speed": 0.5},
        # 256 uneven 2D scenes stepped as one batch (9.7 M particles), replayed as a captured graph
        {"name": "batch_2d_f32", "path": "batch", "scenes": 256, "cells_min": 64, "cells_max": 512,
         "n_min": 2000, "n_max": 200000, "basis": "quadratic", "dtype": "f32", "variant": 10, "steps": 8,
         "reorder": 0.85},
        # one iteration of the inverse problem: rollout with checkpoints, then its pullback (132,651 particles)
        {"name": "inverse_3d_f32", "path": "inverse", "scene": "cube", "cells": 64, "basis": "quadratic",
         "dtype": "f32", "layout": "julia", "steps": 40, "every": 10, "speed": 0.25},
        # the block partition of particles stored in no order (update!(partition, x))
        {"name": "partition_3d_f32", "path": "partition", "scene": "drop", "cells": 128, "dtype": "f32",
         "layout": "julia", "block_log2": 2, "speed": 0.0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["steps", "steps", "steps", "steps", "steps", "calls", "calls", "g2p2g", "batch", "inverse",
                       "partition"])
    dtype = rng.choice(["f32", "f64"])
    layout = rng.choice(["julia", "julia", "soa"])
    if path == "steps":
        scene = rng.choice(["disks", "drop", "drop", "rod", "sphere", "box"])
        c = {"path": path, "scene": scene, "dtype": dtype, "layout": layout, "reorder": rng.choice([0.0, 0.85])}
        if scene == "disks":
            c.update(cells=_log_uniform(rng, 30, 700), basis=rng.choice(["linear", "quadratic", "cubic"]),
                     steps=rng.randint(1, 60), speed=round(rng.uniform(0.02, 0.3), 3))
        elif scene == "drop":
            c.update(cells=_log_uniform(rng, 20, 180 if dtype == "f32" else 130),
                     basis=rng.choice(["linear", "quadratic", "quadratic", "cubic", "ugimp"]),
                     steps=rng.randint(1, 8), speed=round(rng.uniform(0.0, 3.0), 3))
        elif scene == "rod":
            c.update(cells=rng.randint(4, 13), dtype="f64", basis=rng.choice(["kc_quadratic", "quadratic", "kc_cubic"]),
                     steps=rng.randint(1, 6), speed=round(rng.uniform(50.0, 227.0), 2))
        elif scene == "sphere":
            c.update(cells=_log_uniform(rng, 32, 170), dtype="f32", layout="julia", reorder=0.85,
                     basis=rng.choice(["quadratic", "cubic", "ugimp"]), steps=rng.randint(2, 6),
                     speed=round(rng.uniform(0.1, 1.0), 3))
        else:
            b = rng.choice(["wls_quadratic", "quadratic", "kc_quadratic"])
            c.update(cells=_log_uniform(rng, 40, 500), ppc=rng.randint(2, 9), basis=b, steps=rng.randint(1, 8),
                     speed=round(rng.uniform(0.0, 0.5), 3))
        return c
    if path == "calls":
        scene = rng.choice(["box", "drop"])
        c = {"path": path, "scene": scene, "layout": "julia", "stored": rng.random() < 0.5, "dtype": dtype,
             "basis": rng.choice(["linear", "quadratic", "quadratic", "cubic"])}
        if scene == "box":
            c.update(cells=_log_uniform(rng, 40, 600), ppc=rng.randint(2, 9), speed=round(rng.uniform(0.0, 0.5), 3))
        else:
            c.update(cells=_log_uniform(rng, 20, 128), speed=round(rng.uniform(0.0, 3.0), 3))
        return c
    if path == "g2p2g":
        return {"path": path, "scene": "drop", "cells": _log_uniform(rng, 20, 160),
                "basis": rng.choice(["quadratic", "cubic"]),
                "dtype": "f32", "layout": layout, "steps": rng.randint(1, 8), "reorder": rng.choice([0.0, 0.85]),
                "speed": round(rng.uniform(0.0, 2.0), 3)}
    if path == "batch":
        lo = rng.randint(16, 64)
        return {"path": path, "scenes": rng.randint(3, 160), "cells_min": lo, "cells_max": rng.randint(2 * lo, 512),
                "n_min": rng.randint(300, 3000), "n_max": rng.randint(5000, 120000), "basis": "quadratic",
                "dtype": dtype, "variant": rng.choice([0, 2, 10]), "steps": rng.randint(2, 12),
                "reorder": rng.choice([0.0, 0.85])}
    if path == "inverse":
        steps = rng.randint(8, 40)
        return {"path": path, "scene": "cube", "cells": rng.randint(20, 64), "basis": "quadratic", "dtype": dtype,
                "layout": "julia", "steps": steps, "every": rng.randint(3, 20),
                "speed": round(rng.uniform(0.0, 0.5), 3)}
    return {"path": "partition", "scene": "drop", "cells": _log_uniform(rng, 20, 220), "dtype": dtype,
            "layout": "julia", "block_log2": rng.randint(0, 3), "speed": 0.0}


# ---- scenes: particle positions, velocities and strains drawn from the seed, on the GPU ----

def _rand(gen, *shape):
    return torch.rand(*shape, device=DEV, dtype=F64, generator=gen)


def _lattice(*axes):
    """Points of a lattice, first axis fastest."""
    g = torch.meshgrid(*[torch.as_tensor(a, device=DEV, dtype=F64) for a in axes], indexing="ij")
    return torch.stack([a.permute(*reversed(range(a.dim()))).reshape(-1) for a in g], dim=1)


def _axis(lo, hi, s):
    k = int(math.floor((hi - lo) / s - 0.5 + 1e-9)) + 1
    return lo + (torch.arange(k, dtype=F64) + 0.5) * s


def _scene(case, seed):
    """(mesh, params, x, v, strain amplitude, particle length or None) of the case's scene, Float64 on the GPU."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 7919 + 17)
    dt_, name, cells, speed = _dtype(case), case["scene"], case["cells"], case.get("speed", 0.0)
    if name == "disks":
        h = 1.0 / cells
        mesh = th.CartesianMesh(h, (0, 1), (0, 1), dtype=dt_)
        s = h / 2
        pts = _lattice(_axis(0, 1, s), _axis(0, 1, s))
        r = 0.2
        keep = ((pts - r).norm(dim=1) < r) | ((pts - (1 - r)).norm(dim=1) < r)
        x = pts[keep]
        x = (x + (_rand(gen, len(x), 2) - 0.5) * (0.2 * s)).clamp(1e-3 * h, 1 - 1e-3 * h)
        v = torch.where(x[:, :1] > 0.5, -speed, speed) * torch.ones(1, 2, device=DEV, dtype=F64)
        V0 = 1.0 / len(pts)
        prm = th.MPMParams(dt=1e-3 * min(1.0, 100.0 / cells), E=500.0, nu=0.3, rho0=1e3, V0=V0, slip_walls=0b1111)
        return mesh, prm, x, v, 0.02, None
    if name == "drop":
        dx = 1.0 / cells
        mesh = th.CartesianMesh(dx, (0, 1), (0, 1), (0, 1), dtype=dt_, block_size_log2=case.get("block_log2", 2))
        s = dx / 2
        x = _lattice(_axis(0.25, 0.75, s), _axis(0.25, 0.75, s), _axis(0.5, 0.9, s))
        x = x + (_rand(gen, len(x), 3) * 2 - 1) * (0.1 * dx)
        v = torch.zeros_like(x)
        v[:, 2] = -speed
        prm = th.MPMParams(dt=5e-5, E=1e6, nu=0.3, rho0=1e3, V0=s ** 3,
                           gravity=(0.0, 0.0, -9.81), slip_walls=0b111111)
        return mesh, prm, x, v, 0.02, dx / 2
    if name == "rod":
        R, length = 0.0032, 0.0324
        h = R / cells
        mesh = th.CartesianMesh(h, (-3 * R, 3 * R), (-3 * R, 3 * R), (0, 1.1 * length), dtype=dt_)
        s = h / 3
        kr = int(math.floor(R / s))
        ax = (torch.arange(-kr, kr, dtype=F64) + 0.5) * s
        az = (torch.arange(int(math.floor(length / s)), dtype=F64) + 0.5) * s
        x = _lattice(ax, ax, az)
        x = x[(x[:, 0] ** 2 + x[:, 1] ** 2) < R * R]
        x = x + (_rand(gen, len(x), 3) * 2 - 1) * (0.1 * s)
        E, nu, rho0 = 117e9, 0.35, 8.93e3
        lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        dt = 0.8 * h / (math.sqrt((lam + 2 * mu) / rho0) + speed)
        v = torch.zeros_like(x)
        v[:, 2] = -speed
        prm = th.MPMParams(dt=dt, E=E, nu=nu, rho0=rho0, V0=math.pi * R * R * length / len(x), slip_walls=1 << 4)
        return mesh, prm, x, v, 0.002, None
    if name == "sphere":
        dx = 1.0 / cells
        mesh = th.CartesianMesh(dx, (0, 1), (0, 1), (0, 1), dtype=dt_, block_size_log2=3)
        s = dx / 2
        k0, k1 = int(math.floor(0.2 / s - 0.5)), int(math.ceil(0.8 / s - 0.5))
        ax = (torch.arange(k0, k1 + 1, dtype=F64) + 0.5) * s
        parts = []
        for z in ax.split(32):
            p = _lattice(ax, ax, z)
            parts.append(p[((p - 0.5) ** 2).sum(dim=1) < 0.09])
        x = torch.cat(parts)
        x = x + (_rand(gen, len(x), 3) * 2 - 1) * (0.05 * s)
        v = torch.stack([-(x[:, 1] - 0.5), x[:, 0] - 0.5, torch.zeros_like(x[:, 0])], dim=1) * (2.0 * speed)
        v = v + 0.05 * torch.randn(len(x), 3, device=DEV, dtype=F64, generator=gen)
        prm = th.MPMParams(dt=5e-5, E=5e5, nu=0.35, rho0=1e3, V0=s ** 3)
        return mesh, prm, x, v, 0.02, dx / 2
    if name == "cube":
        dx = 1.0 / cells
        mesh = th.CartesianMesh(dx, (0, 1), (0, 1), (0, 1), dtype=dt_)
        s = dx / 2
        ax = _axis(0.3, 0.7, s)
        x = _lattice(ax, ax, ax)
        x = x + (_rand(gen, len(x), 3) * 2 - 1) * (0.05 * s)
        v = 0.05 * torch.randn(len(x), 3, device=DEV, dtype=F64, generator=gen)
        v[:, 0] += speed
        prm = th.MPMParams(dt=2e-4, E=1e5, nu=0.3, rho0=1e3, V0=s ** 3)
        return mesh, prm, x, v, 0.0, None
    # "box": a 2D box of particles at random places, as a program with particle seeding makes it
    h = 1.0 / cells
    mesh = th.CartesianMesh(h, (0, 1), (0, 1), dtype=dt_)
    n = int(0.64 * cells * cells * case["ppc"])
    x = 0.1 + 0.8 * _rand(gen, n, 2)
    v = (_rand(gen, n, 2) - 0.5) * (2 * speed)
    prm = th.MPMParams(dt=0.2 * h / 2.0, E=1e3, nu=0.3, rho0=1e3, V0=0.64 / n, gravity=(0.0, -9.81), slip_walls=0b1111)
    return mesh, prm, x, v, 0.02, None


def _strained(n, d, amp, seed):
    """Deformation gradients of a body under a uniform strain of about ``amp``, column-major."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 104729 + 5)
    eye = torch.eye(d, device=DEV, dtype=F64).reshape(1, d * d)
    return (eye + amp * (2 * _rand(gen, 1, d * d) - 1) - amp * eye).repeat(n, 1)


def _stress(F, prm, d):
    """Neo-Hookean Cauchy stress (column-major, symmetric) and volume of F."""
    M = F.reshape(-1, d, d).transpose(1, 2)
    J = _det(M)
    eye = torch.eye(d, device=F.device, dtype=F.dtype)
    s = prm.mu * (M @ M.transpose(1, 2).contiguous() - eye) + prm.lam * torch.log(J)[:, None, None] * eye
    s = s / J[:, None, None]
    return s.transpose(1, 2).reshape(-1, d * d), prm.V0 * J


def _det(M):
    if M.shape[-1] == 2:
        return M[:, 0, 0] * M[:, 1, 1] - M[:, 0, 1] * M[:, 1, 0]
    return (M[:, 0, 0] * (M[:, 1, 1] * M[:, 2, 2] - M[:, 1, 2] * M[:, 2, 1])
            - M[:, 0, 1] * (M[:, 1, 0] * M[:, 2, 2] - M[:, 1, 2] * M[:, 2, 0])
            + M[:, 0, 2] * (M[:, 1, 0] * M[:, 2, 1] - M[:, 1, 1] * M[:, 2, 0]))


def _inputs(case, seed):
    """(mesh, params, state) with the state's fields in the case's scalar type, (n, components)."""
    mesh, prm, x, v, amp, l = _scene(case, seed)
    dt_ = _dtype(case)
    F = _strained(len(x), mesh.dim, amp, seed).to(dt_).to(F64)
    sigma, V = _stress(F, prm, mesh.dim)
    st = {"x": x.to(dt_), "v": v.to(dt_), "F": F.to(dt_), "sigma": sigma.to(dt_), "V": V.to(dt_),
          "grad_v": torch.zeros(len(x), mesh.dim ** 2, device=DEV, dtype=dt_)}
    if case.get("basis") == "ugimp":
        st["l"] = torch.full((len(x),), l, device=DEV, dtype=dt_)
    return mesh, prm, st


def _fill(P, st):
    for k, t in st.items():
        P.set(k, t)


_FIELDS = ("x", "v", "V", "grad_v", "F", "sigma")


def _grid_fields(case):
    """What a program reads of the grid: after one pass of calls every field; after a loop of steps, which overwrites
    the grid at each of them, its mass and momentum."""
    return th.Grid.FIELDS if case["path"] == "calls" else ("m", "mv")


def _batch_inputs(case, seed):
    """Per-scene (mesh, params, slice of the shared arrays) and the shared particle arrays of the batch."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 1000003 + 29)
    dt_ = _dtype(case)
    u = torch.rand(case["scenes"], 8, generator=torch.Generator().manual_seed(11), dtype=F64)  # the case's sizes
    metas, xs, vs = [], [], []
    at = 0
    for s in range(case["scenes"]):
        a = [float(t) for t in u[s]]
        cells = int(round(case["cells_min"] * (case["cells_max"] / case["cells_min"]) ** a[0]))
        n = int(round(case["n_min"] * (case["n_max"] / case["n_min"]) ** a[1]))
        frac, aspect = 0.2 + 0.4 * a[2], math.exp((a[3] - 0.5) * math.log(2.0))
        w = min(math.sqrt(frac * aspect), 0.98)
        hgt = min(frac / w, 0.98)
        x0, y0 = 0.01 + a[4] * (0.98 - w), 0.01 + a[5] * (0.98 - hgt)
        h = 1.0 / cells
        mesh = th.CartesianMesh(h, (0, 1), (0, 1), dtype=dt_)
        r = _rand(gen, n, 4)
        xs.append(torch.stack([x0 + w * r[:, 0], y0 + hgt * r[:, 1]], dim=1))
        # a body thrown across its scene: one velocity, and particles that stir about it
        drift = torch.tensor([0.4 * a[7] - 0.2, 0.2 - 0.4 * a[5]], device=DEV, dtype=F64)
        vs.append(drift + (r[:, 2:4] - 0.5) * 0.04)
        E = math.exp(math.log(1e3) + a[6] * math.log(1e2))
        V0 = w * hgt / n
        probe = th.MPMParams(dt=1.0, E=E, nu=0.3, rho0=1e3, V0=V0)
        dt = 0.1 * h / (math.sqrt((probe.lam + 2 * probe.mu) / 1e3) + 0.3)
        metas.append((mesh, th.MPMParams(dt=dt, E=E, nu=0.3, rho0=1e3, V0=V0), at, at + n))
        at += n
    x, v = torch.cat(xs).to(dt_), torch.cat(vs).to(dt_)
    F = _strained(at, 2, 0.02, seed).to(dt_)
    sigma, V = (torch.cat(t) for t in zip(*[_stress(F[a_:b].double(), p, 2) for _, p, a_, b in metas]))
    z = torch.zeros(at, 4, device=DEV, dtype=dt_)
    return metas, {"x": x, "v": v, "V": V.to(dt_), "grad_v": z, "F": F, "sigma": sigma.to(dt_)}


# ---- the passes -----------------------------------------------------------------------

def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        metas, big = _batch_inputs(case, seed)
        nodes = sum(m.nnodes() for m, _, _, _ in metas)
        dt_ = _dtype(case)
        grid = {k: torch.zeros((nodes,) if k == "m" else (nodes, 2), device=DEV, dtype=dt_) for k in th.Grid.FIELDS}
        members, at = [], 0
        for mesh, prm, a, b in metas:
            P = th.Particles(0, 2, dt_)
            P.n = b - a
            P.tensors.update({k: t[a:b] for k, t in big.items()})
            G = th.Grid(mesh)
            G.tensors = {k: t[at:at + mesh.nnodes()] for k, t in grid.items()}
            at += mesh.nnodes()
            members.append((G, P, prm))
        batch = th.Batch(members, _basis(case["basis"]), ctx=th.Context())
        batch.set_reorder(case["reorder"])
        batch.set_variant(case["variant"])
        return {"case": case, "batch": batch, "big": big, "grid": grid}
    if path == "partition":
        mesh, prm, x, _, _, _ = _scene(case, seed)
        gen = torch.Generator(device=DEV)
        gen.manual_seed(int(seed) + 11)
        x = x[torch.randperm(len(x), device=DEV, generator=gen)].to(_dtype(case)).contiguous()
        return {"case": case, "x": x, "partition": th.Partition(mesh)}
    mesh, prm, st = _inputs(case, seed)
    n, d = len(st["x"]), mesh.dim
    P = th.Particles(n, d, _dtype(case), layout=case["layout"], with_l="l" in st, with_logE=path == "inverse")
    _fill(P, st)
    sparse = case["scene"] == "sphere"
    G = th.generate_grid(th.SpArray, mesh) if sparse else th.generate_grid(mesh, layout=case["layout"])
    s = {"case": case, "mesh": mesh, "prm": prm, "P": P, "G": G, "basis": _basis(case["basis"]), "ctx": th.Context()}
    if path == "calls":
        s["W"] = th.generate_basis_weights(s["basis"], mesh, n, deferred=not case["stored"])
    elif path == "g2p2g":
        th.P2G(G, P, s["basis"], prm, ctx=s["ctx"])
    elif path == "inverse":
        s["start"] = {k: P.tensors[k].clone() for k in ("x", "v", "F", "V", "sigma")}
        s["target"] = st["x"].double() + torch.tensor([0.1, 0.0, 0.0], device=DEV, dtype=F64)
        s["adj"] = th.Adjoint(n, d)
    return s


def run(s):
    case, path = s["case"], s["case"]["path"]
    if path == "batch":
        s["batch"].step(case["steps"])
        return {"particles": dict(s["big"]), "grid": {k: s["grid"][k] for k in _grid_fields(case)}}
    if path == "partition":
        p = th.update(s["partition"], s["x"])
        return {"particleindices": p.particleindices, "starts": p.starts, "stops": p.stops, "nassigned": p.nassigned}
    P, G, prm, basis, ctx = s["P"], s["G"], s["prm"], s["basis"], s["ctx"]
    if path == "steps":
        th.step(G, P, basis, prm, nsteps=case["steps"], reorder_threshold=case["reorder"], ctx=ctx)
    elif path == "calls":
        th.update(s["W"], P, s["mesh"], ctx=ctx)
        th.P2G(G, P, s["W"], prm, ctx=ctx)
        th.G2P(G, P, s["W"], prm, ctx=ctx)
    elif path == "g2p2g":
        th.g2p2g_steps(G, P, basis, prm, nsteps=case["steps"], reorder_threshold=case["reorder"], ctx=ctx)
    else:
        # from the initial state: rollout, the loss mean|x(T) - target|^2, its gradient in the parameters' own type
        for k, t in s["start"].items():
            P.tensors[k].copy_(t)
        th.rollout(G, P, basis, prm, case["steps"], checkpoint_every=case["every"], ctx=ctx)
        adj = s["adj"]
        diff = P.tensors["x"].double() - s["target"]
        torch.mul(diff, 2.0 / len(diff), out=adj.x)
        adj.v.zero_()
        adj.F.zero_()
        adj.logE.zero_()
        th.rollout_adjoint(G, basis, prm, adj, ctx=ctx)
        return {"x": P.x, "v": P.v, "F": P.F, "grad_v0": adj.v.to(P.dtype)}
    return {"particles": {k: P.tensors[k] for k in _FIELDS}, "grid": {k: G.tensors[k] for k in _grid_fields(case)}}


def _count(case):
    """Particles of the case, without making them."""
    if case["path"] == "batch":
        r = math.log(case["n_max"] / case["n_min"])
        return int(case["scenes"] * (case["n_max"] - case["n_min"]) / max(r, 1e-9))  # mean of a log-uniform draw
    c, name = case["cells"], case["scene"]
    if name == "disks":
        return int(math.pi * 0.04 * 2 * 4 * c * c)
    if name == "drop":
        return int(0.1 * 8 * c ** 3)
    if name == "rod":
        return int(math.pi * (3 * c) ** 2 * (0.0324 / 0.0032) * 3 * c)
    if name == "sphere":
        return int(4 / 3 * math.pi * 0.027 * 8 * c ** 3)
    if name == "cube":
        return int((0.8 * c) ** 3)
    return int(0.64 * c * c * case["ppc"])


def work(case):
    n, s = _count(case), 4 if case["dtype"] == "f32" else 8
    if case["path"] == "partition":
        nb = ((case["cells"] >> case["block_log2"]) + 1) ** 3
        return {"bytes": n * (3 * s + 4) + 8 * nb, "flops": 6 * n}
    d = 2 if case["path"] == "batch" or case["scene"] in ("disks", "box") else 3
    ppc = {"disks": 4, "box": case.get("ppc", 1), "rod": 27}.get(case.get("scene"), 8)
    if case["path"] == "batch":
        cells = (case["cells_max"] - case["cells_min"]) / math.log(case["cells_max"] / case["cells_min"])
        ppc = n / (case["scenes"] * 0.4 * cells * cells)
    name = case["basis"].split("_")[-1]
    width = {"linear": 2, "quadratic": 3, "cubic": 4, "ugimp": 3}[name]
    K, nodes = width ** d, n / ppc
    # one step: the particle state and the active nodes once through P2G and once through G2P
    bytes_step = s * ((5 * d * d + 6 * d + 2) * n + (8 * d + 2) * nodes)
    flops_step = n * K * (2 + 6 * d + 4 * d * d)
    if case["path"] == "calls":
        extra = n * (K * (1 + d) * s + 2 * d * 8) * 3 if case["stored"] else 0  # weights written once, read twice
        return {"bytes": bytes_step + extra, "flops": flops_step}
    if case["path"] == "inverse":
        # the forward, its replay, and the reversal (particle adjoints in and out, the forward grid, Float64)
        back = 8 * n * 2 * (2 * d + d * d) + s * n * (3 * d + 2 * d * d) + (s + 8) * nodes * (1 + 3 * d)
        return {"bytes": case["steps"] * (2 * bytes_step + back), "flops": case["steps"] * 5 * flops_step}
    return {"bytes": case["steps"] * bytes_step, "flops": case["steps"] * flops_step}


# ---- the same passes in Float64 torch ----------------------------------------------------

def _kernel1d(name, xi, l):
    """Value and derivative of the 1-D kernel at the normalised offset xi."""
    s = torch.where(torch.signbit(xi), -1.0, 1.0).to(xi.dtype)
    a = xi.abs()
    z = torch.zeros_like(a)
    if name == "linear":
        return torch.where(a < 1, 1 - a, z), torch.where(a < 1, -s, z)
    if name == "quadratic":
        u = 1.5 - a
        return (torch.where(a < 0.5, 0.75 - a * a, torch.where(a < 1.5, u * u / 2, z)),
                torch.where(a < 0.5, -2 * a * s, torch.where(a < 1.5, -u * s, z)))
    if name == "cubic":
        u = 2 - a
        return (torch.where(a < 1, 2 / 3 - a * a + a ** 3 / 2, torch.where(a < 2, u ** 3 / 6, z)),
                torch.where(a < 1, (-2 * a + 1.5 * a * a) * s, torch.where(a < 2, -u * u / 2 * s, z)))
    u = 1 + l / 2 - a
    return (torch.where(a < l / 2, 1 - (4 * a * a + l * l) / (4 * l),
                        torch.where(a < 1 - l / 2, 1 - a, torch.where(a < 1 + l / 2, u * u / (2 * l), z))),
            torch.where(a < l / 2, -2 * a * s / l,
                        torch.where(a < 1 - l / 2, -s, torch.where(a < 1 + l / 2, -u * s / l, z))))


def _weights(mesh, name, x, l):
    """Node indices (n, K), values (n, K) and gradients (n, K, d) of the particles' windows; zero off the mesh."""
    d = mesh.dim
    corr, kern = (name.split("_") + [None])[:2] if "_" in name else ("", name)
    width = {"linear": 2, "quadratic": 3, "cubic": 4, "ugimp": 3}[kern]
    val, der, off, ok, idx = [], [], [], [], []
    inside = torch.ones(len(x), dtype=torch.bool, device=x.device)
    full = torch.ones_like(inside)
    for c in range(d):
        xi = (x[:, c] - mesh.xmin[c]) / mesh.h
        with torch.no_grad():
            f = torch.floor(xi)
            inside &= (f >= 0) & (f <= mesh.dims[c] - 2)
            if kern == "ugimp":
                lo = torch.floor(xi - (1 + l / 2)) + 1
                last = torch.floor(xi + (1 + l / 2))
            else:
                lo = torch.floor(xi - (width - 2) / 2)
                last = lo + width - 1
            i = lo[:, None] + torch.arange(width, device=x.device, dtype=F64)
            good = (i >= 0) & (i <= mesh.dims[c] - 1) & (i <= last[:, None])
            full &= good.all(dim=1) if kern != "ugimp" else ((lo >= 0) & (last <= mesh.dims[c] - 1))
        o = xi[:, None] - i
        v, g = _kernel1d(kern, o, None if l is None else l[:, None])
        val.append(v * good)
        der.append(g * good / mesh.h)
        off.append(-o)
        ok.append(good)
        idx.append(i.clamp(0, mesh.dims[c] - 1).long())
    n, K = len(x), width ** d
    sh = [(n,) + (1,) * (d - 1 - c) + (width,) + (1,) * c for c in range(d)]  # first axis fastest
    w = inside.to(F64).reshape((n,) + (1,) * d)
    lin, stride = 0, 1
    g = [w] * d
    for c in range(d):
        w = w * val[c].reshape(sh[c])
        g = [g[e] * (der[c] if e == c else val[c]).reshape(sh[c]) for e in range(d)]
        lin = lin + idx[c].reshape(sh[c]) * stride
        stride *= mesh.dims[c]
    w, g, lin = w.reshape(n, K), torch.stack([t.reshape(n, K) for t in g], dim=2), lin.expand(w.shape).reshape(n, K)
    if corr:
        # the moment fit (offsets in cells): every particle for WLS, those with a cut window for KernelCorrection
        pick = (inside if corr == "wls" else inside & ~full).nonzero()[:, 0]
        if len(pick):
            o = [off[c][pick].reshape((len(pick),) + sh[c][1:]) for c in range(d)]
            terms = [torch.ones((len(pick),) + (width,) * d, device=x.device, dtype=F64)]
            terms += [t.expand(terms[0].shape) for t in o]
            if corr == "kc":
                terms += [(o[0] * o[1]).expand(terms[0].shape)]
                if d == 3:
                    terms += [(o[0] * o[2]).expand(terms[0].shape), (o[1] * o[2]).expand(terms[0].shape)]
                    terms += [o[0] * o[1] * o[2]]
            Pm = torch.stack([t.reshape(len(pick), K) for t in terms], dim=1)  # (n, terms, K)
            N = w[pick]
            A = (Pm * N[:, None, :]) @ Pm.transpose(1, 2).contiguous()
            Q = _solve(A, Pm)  # M^-1 P(x_i - x_p)
            w = w.index_copy(0, pick, N * Q[:, 0])
            g = g.index_copy(0, pick, (N[:, None, :] * Q[:, 1:d + 1]).transpose(1, 2) / mesh.h)
    return lin, w, g


def _solve(A, B):
    """A^-1 B of small symmetric positive definite systems by Gauss-Jordan elimination."""
    A, B = A.clone(), B.clone()
    for k in range(A.shape[1]):
        p = A[:, k:k + 1, k:k + 1]
        row, rb = A[:, k:k + 1] / p, B[:, k:k + 1] / p
        f = A[:, :, k:k + 1].clone()
        f[:, k] = 0
        A, B = A - f * row, B - f * rb
        A[:, k:k + 1], B[:, k:k + 1] = row, rb
    return B


def _chunks(n, K):
    size = max(1, 24_000_000 // K)
    return [(a, min(n, a + size)) for a in range(0, n, size)]


def _p2g(mesh, name, prm, S, x, l, weights=None):
    """Grid m, mv, f, vn, v of the state S with the weights at x."""
    d, N = mesh.dim, mesh.nnodes()
    out = torch.zeros(N, 1 + 2 * d, device=x.device, dtype=F64)
    width = 4 if "cubic" in name else 2 if "linear" in name else 3
    for a, b in _chunks(len(x), width ** d):
        lin, w, g = weights or _weights(mesh, name, x[a:b], None if l is None else l[a:b])
        sig = S["sigma"][a:b].reshape(-1, d, d).transpose(1, 2)
        fp = (-S["V"][a:b, None, None] * g) @ sig.transpose(1, 2).contiguous()
        cols = torch.cat([(w * prm.mp)[:, :, None], w[:, :, None] * (prm.mp * S["v"][a:b])[:, None, :], fp], dim=2)
        out = out.index_add(0, lin.reshape(-1), cols.reshape(-1, 1 + 2 * d))
    m, mv, f = out[:, 0], out[:, 1:1 + d], out[:, 1 + d:]
    has = m > 0
    minv = torch.where(has, 1 / torch.where(has, m, torch.ones_like(m)), torch.zeros_like(m))
    vn = mv * minv[:, None]
    grav = torch.tensor(list(prm.gravity)[:d], device=x.device, dtype=F64)
    v = vn + (f * minv[:, None] + has[:, None] * grav) * prm.dt
    I = torch.arange(N, device=x.device)
    keep = torch.ones(N, d, device=x.device, dtype=F64)
    for c in range(d):
        i = I % mesh.dims[c]
        I = I // mesh.dims[c]
        if (prm.slip_walls >> (2 * c)) & 1:
            keep[:, c] *= (i != 0)
        if (prm.slip_walls >> (2 * c + 1)) & 1:
            keep[:, c] *= (i != mesh.dims[c] - 1)
    return {"m": m, "mv": mv, "f": f, "vn": vn, "v": v * keep}


def _g2p(mesh, name, prm, G, S, l, weights=None):
    """The state after @G2P."""
    d = mesh.dim
    width = 4 if "cubic" in name else 2 if "linear" in name else 3
    got = {k: [] for k in _FIELDS}
    for a, b in _chunks(len(S["x"]), width ** d):
        x = S["x"][a:b]
        lin, w, g = weights or _weights(mesh, name, x, None if l is None else l[a:b])
        vi, vni = G["v"][lin], G["vn"][lin]
        L = vi.transpose(1, 2) @ g.contiguous()  # L[r, c] = sum v_r dw_c
        F = S["F"][a:b].reshape(-1, d, d).transpose(1, 2)
        F = F + prm.dt * (L @ F.contiguous())
        Fc = F.transpose(1, 2).reshape(-1, d * d)
        sig, V = _stress(Fc, prm, d)
        got["x"].append(x + (w[:, :, None] * vi).sum(dim=1) * prm.dt)
        got["v"].append(S["v"][a:b] + (w[:, :, None] * (vi - vni)).sum(dim=1))
        got["grad_v"].append(L.transpose(1, 2).reshape(-1, d * d))
        got["F"].append(Fc)
        got["sigma"].append(sig)
        got["V"].append(V)
    return {k: torch.cat(t) for k, t in got.items()}


def _laid_out(case, S, G):
    """The pass's outputs from the Float64 state and grid; a loop that reorders its particles stores them in an order
    of the engine's own, so only its grid is given."""
    soa = case.get("layout") == "soa"
    t = lambda a: a.t().contiguous() if soa and a.dim() == 2 else a  # noqa: E731
    return {"particles": {k: None if case.get("reorder") else t(S[k]) for k in _FIELDS},
            "grid": {k: t(G[k]) for k in _grid_fields(case)}}


def exact(case, seed):
    path = case["path"]
    if path == "partition":
        return None  # whole numbers
    if case.get("scene") == "sphere":
        return None  # storage order of the particles and of the sparse grid is the engine's
    if path == "batch":
        metas, big = _batch_inputs(case, seed)
        parts, grids = [], []
        for mesh, prm, a, b in metas:
            S = {k: t[a:b].double() for k, t in big.items()}
            for _ in range(case["steps"]):
                G = _p2g(mesh, case["basis"], prm, S, S["x"], None)
                S = _g2p(mesh, case["basis"], prm, G, S, None)
            parts.append(S)
            grids.append(G)
        return {"particles": {k: None if case["reorder"] else torch.cat([p[k] for p in parts]) for k in _FIELDS},
                "grid": {k: torch.cat([g[k] for g in grids]) for k in _grid_fields(case)}}
    mesh, prm, st = _inputs(case, seed)
    S = {k: t.double() for k, t in st.items()}
    l = S.pop("l") / mesh.h if "l" in S else None
    name = case["basis"]
    if path == "inverse":
        return _exact_inverse(case, mesh, prm, S)
    steps = case.get("steps", 1)
    if path == "g2p2g":
        G = _p2g(mesh, name, prm, S, S["x"], l)
        for _ in range(steps):
            x = S["x"]
            S = _g2p(mesh, name, prm, G, S, l)
            G = _p2g(mesh, name, prm, S, x, l)
    else:
        for _ in range(steps):
            G = _p2g(mesh, name, prm, S, S["x"], l)
            S = _g2p(mesh, name, prm, G, S, l)
    return _laid_out(case, S, G)


def _exact_inverse(case, mesh, prm, S):
    from torch.utils.checkpoint import checkpoint

    name, target = case["basis"], S["x"] + torch.tensor([0.1, 0.0, 0.0], device=DEV, dtype=F64)
    x, v, F = (S[k].clone().requires_grad_() for k in ("x", "v", "F"))

    def one(x, v, F):
        sig, V = _stress(F, prm, 3)
        lin, w, g = _weights(mesh, name, x, None)
        state = {"x": x, "v": v, "F": F, "sigma": sig, "V": V}
        G = _p2g(mesh, name, prm, state, x, None, (lin, w, g))
        T = _g2p(mesh, name, prm, G, state, None, (lin, w, g))
        return T["x"], T["v"], T["F"]

    cur = (x, v, F)
    for _ in range(case["steps"]):
        cur = checkpoint(one, *cur, use_reentrant=False)
    loss = ((cur[0] - target) ** 2).sum() / len(x)
    gv, = torch.autograd.grad(loss, (v,))
    return {"x": cur[0].detach(), "v": cur[1].detach(), "F": cur[2].detach(), "grad_v0": gv}

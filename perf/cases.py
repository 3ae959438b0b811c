"""The work that is timed: one-step building blocks of a FLIP multiphase run.

Each case is one pass through the public entry points (the C ABI of
include/mpflip.h and the `Simulator` class over it) on device-resident data,
at the sizes of the library's own scenes (64^3 to 256^3 cells, 8 particles per
cell) and at ragged sizes between them:

  sort      mpf_hash_sort_noalloc on caller buffers (the sort of a serving loop)
  project   face velocities in, one pressure projection, face velocities out,
            in the three precision forms, with and without air and solids
  transfer  P2G of both phases, extrapolation with the wall rules, G2P
  surface   level set from the particles, then the marching-cubes mesh
  correct   sort, spring position correction, and the sort after it
  heat      heat transfer to the grid, the implicit diffusion, and back
  adjoint   the reverse of G2P, extrapolation and P2G (FP64 cotangents)
  step      a whole mpf_step from a given particle state

The particles of a state lie in the order of an earlier sort and have moved
since, so cells hold 8 on average, not exactly; velocities are smooth with a
small random part.  torch is imported before the package, so that the library
and torch share one HIP runtime and the library takes torch's device memory.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

mp = importlib.import_module("2017multiphase_amd")

H = 1.0 / 64
FACES = ["WATER_UX", "WATER_UY", "WATER_UZ", "AIR_UX", "AIR_UY", "AIR_UZ"]
DEV = "cuda"


def listed():
    return [
        # a small coupled tool that sorts its own points: launches and latency
        {"name": "sort_ragged_small", "kind": "sort", "nx": 33, "ny": 47, "nz": 29, "fill": 0.7},
        # bubble_rise scene: plain FP32 form, an air sphere in 60% water
        {"name": "project_fp32_64", "kind": "project", "nx": 64, "ny": 64, "nz": 64, "fill": 0.6, "precision": mp.FP32,
         "tol": 1e-6, "bubbles": 1, "rmin": 0.12, "rmax": 0.13, "solids": 0, "rho_air": 1.0},
        # diff_slab scene: the all-FP64 form that gradients are checked with
        {"name": "project_fp64_96", "kind": "project", "nx": 96, "ny": 96, "nz": 96, "fill": 0.42, "precision": mp.FP64,
         "tol": 1e-6, "bubbles": 6, "rmin": 0.04, "rmax": 0.1, "solids": 0, "rho_air": 1.0},
        # bubble_column scene at half its size: many bubbles, tight tolerance
        {"name": "project_mixed_192", "kind": "project", "nx": 192, "ny": 192, "nz": 192, "fill": 0.85,
         "precision": mp.MIXED, "tol": 1e-8, "bubbles": 128, "rmin": 0.008, "rmax": 0.031, "solids": 0,
         "rho_air": 1.0},
        # melt_freeze scene: liquid with solid blocks, the benchmark's size
        {"name": "project_mixed_256", "kind": "project", "nx": 256, "ny": 256, "nz": 256, "fill": 0.68,
         "precision": mp.MIXED, "tol": 1e-6, "bubbles": 0, "solids": 4, "rho_air": 1.0},
        # particle-grid transfers of a mid-size two-phase scene
        {"name": "transfer_128", "kind": "transfer", "nx": 128, "ny": 128, "nz": 128, "fill": 0.7, "bubbles": 8,
         "rmin": 0.02, "rmax": 0.08, "flip": 0.95},
        # an output frame: the surface of the liquid as a mesh
        {"name": "surface_128", "kind": "surface", "nx": 128, "ny": 128, "nz": 128, "fill": 0.7, "bubbles": 8,
         "rmin": 0.02, "rmax": 0.08},
        # particle spacing after advection, on a ragged grid
        {"name": "correct_ragged", "kind": "correct", "nx": 121, "ny": 99, "nz": 150, "fill": 0.66, "bubbles": 4,
         "rmin": 0.02, "rmax": 0.08},
        # heated liquid of the boiling scene
        {"name": "heat_128", "kind": "heat", "nx": 128, "ny": 128, "nz": 128, "fill": 0.7, "solids": 2, "jacobi": 1},
        # one reverse step of the differentiable slab scene
        {"name": "adjoint_96", "kind": "adjoint", "nx": 96, "ny": 96, "nz": 96, "fill": 0.42, "bubbles": 6,
         "rmin": 0.04, "rmax": 0.1},
        # whole steps: the boiling scene at its own size, the benchmark's scene
        {"name": "step_boiling_128", "kind": "step", "scene": "boiling", "nx": 128, "ny": 128, "nz": 128, "fill": 0.7,
         "solids": 0, "precision": mp.MIXED},
        {"name": "step_melt_freeze_256", "kind": "step", "scene": "melt_freeze", "nx": 256, "ny": 256, "nz": 256,
         "fill": 0.68, "solids": 4, "precision": mp.MIXED},
    ]


def _size(rng, lo, hi):
    """A grid whose cell count is log-uniform between lo^3 and hi^3, sides within about 1.4 of each other."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    s = [max(12, int(round(n * math.exp(rng.uniform(-0.17, 0.17))))) for _ in range(3)]
    f = n ** 3 / (s[0] * s[1] * s[2])
    s[2] = max(12, int(round(s[2] * f)))
    return {"nx": s[0], "ny": s[1], "nz": s[2]}


def _bubbles(rng, most):
    """Up to `most` bubbles: few large ones or many small ones (radii as fractions of the grid's width)."""
    n = rng.randint(0, most)
    lo = 0.12 / max(1, n) ** 0.5
    return {"bubbles": n, "rmin": round(max(0.008, lo / 2), 4), "rmax": round(max(0.02, lo), 4)}


def draw(rng):
    kind = rng.choice(["sort", "project", "project", "project", "transfer", "surface", "correct", "heat", "adjoint",
                       "step"])
    fill = round(rng.uniform(0.4, 0.85), 3)
    if kind == "sort":
        return {"kind": kind, **_size(rng, 30, 200), "fill": fill}
    if kind == "project":
        prec = rng.choice([mp.FP32, mp.FP64, mp.MIXED, mp.MIXED])
        air = rng.random() < 0.5
        return {"kind": kind, **_size(rng, 48, 200 if prec == mp.MIXED else 144), "fill": fill, "precision": prec,
                "tol": rng.choice([1e-6, 1e-8]) if prec == mp.MIXED else 1e-6, **_bubbles(rng, 64 if air else 0),
                "solids": 0 if air else rng.randint(0, 4), "rho_air": rng.choice([1.0, 5.0])}
    if kind == "transfer":
        return {"kind": kind, **_size(rng, 48, 200), "fill": fill, **_bubbles(rng, 64),
                "flip": rng.choice([0.95, 1.0])}
    if kind in ("surface", "correct"):
        return {"kind": kind, **_size(rng, 48, 200), "fill": fill, **_bubbles(rng, 64)}
    if kind == "heat":
        return {"kind": kind, **_size(rng, 48, 176), "fill": fill, "solids": rng.randint(0, 4),
                "jacobi": int(rng.random() < 0.75)}
    if kind == "adjoint":
        return {"kind": kind, **_size(rng, 48, 112), "fill": fill, **_bubbles(rng, 8)}
    return {"kind": kind, "scene": rng.choice(["boiling", "melt_freeze"]), **_size(rng, 48, 176), "fill": fill,
            "solids": rng.randint(1, 4), "precision": mp.MIXED}


# ---- geometry (torch, from the seed alone) ----
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g, np.random.default_rng(seed)


def _axes(case):
    f = {"device": DEV, "dtype": torch.float32}
    return (torch.arange(case["nx"], **f).view(-1, 1, 1), torch.arange(case["ny"], **f).view(1, -1, 1),
            torch.arange(case["nz"], **f).view(1, 1, -1))


def _geometry(case):
    """liquid, air and solid cell masks, and the air level set (positive inside bubbles, metres).

    They belong to the case (the scene), so that every seed has as many particles."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rng = np.random.default_rng([nx, ny, nz])
    I, J, K = _axes(case)
    inner = (I >= 1) & (I <= nx - 2) & (J >= 1) & (J <= ny - 2) & (K >= 1) & (K <= nz - 2)
    top = case["fill"] * nz
    a = rng.uniform(0.3, 1.0, 2)
    wave = a[0] * torch.sin(I * (2 * math.pi * 2 / nx) + rng.uniform(0, 6)) + a[1] * torch.cos(
        J * (2 * math.pi * 3 / ny) + rng.uniform(0, 6))
    liquid = inner & (K < top + wave)
    ls = torch.full((nx, ny, nz), -1e3, device=DEV)
    for _ in range(case.get("bubbles", 0)):
        r = rng.uniform(case["rmin"], case["rmax"]) * nx
        c = [rng.uniform(r + 2, max(r + 3, s - r - 2)) for s in (nx, ny, top - 1)]
        d = torch.sqrt((I + 0.5 - c[0]) ** 2 + (J + 0.5 - c[1]) ** 2 + (K + 0.5 - c[2]) ** 2)
        ls = torch.maximum(ls, r - d)
    ls = ls * H
    air = liquid & (ls > 0)
    solid = torch.zeros_like(liquid)
    b = max(2, int(round(0.16 * min(nx, ny, top))))
    for _ in range(case.get("solids", 0)):
        lo = [int(rng.integers(2, max(3, s - 2 - b))) for s in (nx, ny, int(top))]
        solid[lo[0]:lo[0] + b, lo[1]:lo[1] + b, lo[2]:lo[2] + b] = True
    solid &= liquid
    return liquid & ~air & ~solid, air & ~solid, solid, ls


def _modes(rng, x, y, z, L):
    """A smooth velocity component: a few sine modes of up to about 1 m/s."""
    u = 0.0
    for _ in range(4):
        kx, ky, kz = rng.integers(1, 5, 3) * (math.pi / np.asarray(L))
        p = rng.uniform(0, 2 * math.pi, 3)
        u = u + rng.uniform(-0.5, 0.5) * torch.sin(kx * x + p[0]) * torch.sin(ky * y + p[1]) * torch.sin(kz * z + p[2])
    return u


def _particles(case, seed):
    """8 particles per occupied cell in cell order, moved since by up to about a third of a cell."""
    gen, rng = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    liquid, air, solid, _ = _geometry(case)
    L = [nx * H, ny * H, nz * H]
    kind = torch.full((nx, ny, nz), -1, device=DEV, dtype=torch.int8)
    kind[liquid] = mp.TYPEFLUID
    kind[air] = mp.TYPEAIR
    kind[solid] = mp.TYPESOLID
    cells = torch.nonzero(kind.view(-1) >= 0).view(-1)
    flag = kind.view(-1)[cells].repeat_interleave(8)
    n = flag.numel()
    cells = cells.repeat_interleave(8)
    pos = torch.rand((n, 3), device=DEV, generator=gen)
    pos[:, 0] += torch.div(cells, ny * nz, rounding_mode="floor")
    pos[:, 1] += torch.div(cells, nz, rounding_mode="floor") % ny
    pos[:, 2] += cells % nz
    pos *= H
    del cells
    vel = torch.empty_like(pos)
    for a in range(3):
        vel[:, a] = _modes(rng, pos[:, 0], pos[:, 1], pos[:, 2], L)
    moving = (flag != mp.TYPESOLID)[:, None]
    step = 4e-3 * vel + (0.05 * H) * torch.randn((n, 3), device=DEV, generator=gen)
    pos += torch.where(moving, step.clamp_(-0.35 * H, 0.35 * H), 0.0)
    for a in range(3):
        pos[:, a].clamp_(1.001 * H, L[a] - 1.001 * H)
    vel += 0.02 * torch.randn((n, 3), device=DEV, generator=gen)
    vel *= moving
    return {"pos": pos, "vel": vel, "flag": flag}, n, gen, rng


def _attributes(parts, n, cfg, gen, t_liquid, t_noise, t_solid, lheat):
    """Mass, temperature, latent heat and gas content as the scenes set them."""
    fluid, solid = parts["flag"] == mp.TYPEFLUID, parts["flag"] == mp.TYPESOLID
    f = {"device": DEV, "dtype": torch.float32}
    parts["mass"] = torch.full((n,), cfg.m0, **f)
    T = t_liquid + t_noise * (2 * torch.rand((n,), generator=gen, **f) - 1)
    parts["T"] = torch.where(solid, torch.full((), t_solid, **f), T)
    parts["lheat"] = torch.where(fluid, torch.full((), lheat, **f), torch.zeros((), **f))
    parts["solubility"] = torch.where(fluid, torch.full((), 0.95 * cfg.airm0, **f), torch.zeros((), **f))
    parts["gascontain"] = 0.88 * parts["solubility"]
    return parts


# ---- C ABI calls on device memory ----
def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _check(sim, status, allow=(mp.OK,)):
    if status not in allow:
        raise mp.MpfError(status, sim.L.mpf_last_error(sim.h).decode())


def _get(sim, name, out):
    _check(sim, sim.L.mpf_get_field(sim.h, mp.FIELD_ID[name], _ptr(out), mp.DEVICE))


def _set(sim, name, t):
    _check(sim, sim.L.mpf_set_field(sim.h, mp.FIELD_ID[name], _ptr(t), mp.DEVICE))


def _get_particles(sim, out):
    n = ctypes.c_int64()
    order = ("pos", "vel", "flag", "mass", "T", "lheat", "solubility", "gascontain")
    _check(sim, sim.L.mpf_get_particles(sim.h, ctypes.byref(n), *[_ptr(out.get(k)) for k in order], mp.DEVICE))


def _face_shapes(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return [(nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)] * 2


def _face_set(case, dtype=torch.float32):
    return [torch.empty(s, device=DEV, dtype=dtype) for s in _face_shapes(case)]


def _table(ts):
    return ctypes.cast((ctypes.c_void_p * 6)(*[t.data_ptr() for t in ts]), ctypes.c_void_p)


def _config(case, **kw):
    return mp.default_config(case["nx"], case["ny"], case["nz"], **kw)


# ---- states ----
def _prepare_sort(case, seed):
    parts, n, _, _ = _particles(case, seed)
    cells = case["nx"] * case["ny"] * case["nz"]
    u = {"device": DEV, "dtype": torch.int32}
    return {"cfg": _config(case), "n": n, "pos": parts["pos"],
            "out": [torch.empty(n, **u), torch.empty(n, **u), torch.empty(cells, **u), torch.empty(cells, **u)]}


def _faces_and_marks(case, seed):
    """Extrapolated face velocities of both phases, cell types and the merged level set."""
    gen, rng = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    liquid, air, solid, ls = _geometry(case)
    mark = torch.full((nx, ny, nz), mp.TYPEVACUUM, device=DEV, dtype=torch.int8)
    mark[liquid] = mp.TYPEFLUID
    mark[air] = mp.TYPEAIR
    mark[solid] = mp.TYPESOLID
    for a in range(3):
        mark.select(a, 0).fill_(mp.TYPEBOUNDARY)
        mark.select(a, mark.shape[a] - 1).fill_(mp.TYPEBOUNDARY)
    edge = mark == mp.TYPEBOUNDARY
    ls = torch.where(edge, -0.5 * H, torch.where(liquid | air, ls.clamp(-2.5 * H, 2.5 * H), 0.5 * H)).float()
    L = [nx * H, ny * H, nz * H]
    faces = []
    for f, shape in enumerate(_face_shapes(case)):
        a = f % 3
        x, y, z = [(torch.arange(shape[d], device=DEV, dtype=torch.float32) + (0.0 if d == a else 0.5)) * H
                   for d in range(3)]
        u = _modes(rng, x.view(-1, 1, 1), y.view(1, -1, 1), z.view(1, 1, -1), L)
        u = u + 0.02 * torch.randn(shape, device=DEV, generator=gen) - (0.0098 if a == 2 else 0.0)
        for w in (0, 1, shape[a] - 2, shape[a] - 1):  # walls
            u.select(a, w).fill_(0.0)
        faces.append(u.float().contiguous())
    return mark, ls, faces


def _prepare_project(case, seed):
    mark, ls, faces = _faces_and_marks(case, seed)
    cfg = _config(case, precision=case["precision"], tol=case["tol"], rho_liquid=1000.0, rho_air=case["rho_air"],
                  max_iters=20000, solid_constraint=1 if case["solids"] else 0, mc_enabled=0, heat_enabled=0,
                  particle_capacity=1024)
    sim = mp.Simulator(cfg)
    torch.cuda.synchronize()
    _set(sim, "MARK", mark)
    _set(sim, "LSMERGE", ls)
    return {"sim": sim, "in": faces, "out": _face_set(case)}


def _sorted_sim(case, seed, t=(293.15, 0.0, 263.15, 10.0), **kw):
    parts, n, gen, rng = _particles(case, seed)
    cfg = _config(case, particle_capacity=n + n // 8 + 1024, **kw)
    _attributes(parts, n, cfg, gen, *t)
    sim = mp.Simulator(cfg)
    torch.cuda.synchronize()
    sim.set_particles(n, where=mp.DEVICE, **parts)
    sim.hash_sort()
    return sim, parts, n, gen, rng


def _prepare_transfer(case, seed):
    sim, _, n, _, _ = _sorted_sim(case, seed, flip_alpha=case["flip"], mc_enabled=0, heat_enabled=0)
    sim.levelset_update()
    sim.synchronize()
    return {"sim": sim, "faces": _face_set(case), "vel": torch.empty((n, 3), device=DEV)}


def _prepare_surface(case, seed):
    cells = (case["nx"], case["ny"], case["nz"])
    most = max(1 << 16, case["nx"] * case["ny"] * case["nz"] // 4)
    sim, _, _, _, _ = _sorted_sim(case, seed, heat_enabled=0, mc_max_verts=most, mc_max_tris=2 * most)
    sim.synchronize()
    # the caller's mesh buffers hold what the configuration allows, used from the front
    return {"sim": sim, "ls": [torch.empty(cells, device=DEV) for _ in range(3)],
            "mark": torch.empty(cells, device=DEV, dtype=torch.int8),
            "verts": torch.zeros((most, 3), device=DEV), "normals": torch.zeros((most, 3), device=DEV),
            "tris": torch.zeros((2 * most, 3), device=DEV, dtype=torch.int32)}


def _prepare_correct(case, seed):
    parts, n, gen, _ = _particles(case, seed)
    cfg = _config(case, particle_capacity=n, mc_enabled=0, heat_enabled=0)
    _attributes(parts, n, cfg, gen, 293.15, 0.0, 293.15, 10.0)
    sim = mp.Simulator(cfg)
    torch.cuda.synchronize()
    return {"sim": sim, "n": n, "in": parts, "pos": torch.empty_like(parts["pos"])}


def _prepare_heat(case, seed):
    sim, _, n, _, _ = _sorted_sim(
        case, seed, (1.05, 0.03, 0.8, 0.1), dt=1e-3, mc_enabled=0, heat_enabled=1,
        heat_solver=mp.HEAT_JACOBI if case["jacobi"] else mp.HEAT_CG, heat_jacobi_iters=10, default_temperature=1.0,
        heat_add_bottom=1, heat_increase_bottom=0.02, heat_bottom_clamp=1.2, heat_extend_boundary=1,
        heat_vacuum_neumann=1, melting_point=1.0, boiling_point=10.0, liquid_heat_th=0.1, temperature0=1.0,
        heat_alpha=[0.18, 0.08, 0.0, 0.0001, 0.08, 0.2], solid_constraint=1 if case["solids"] else 0)
    sim.levelset_update()
    sim.synchronize()
    return {"sim": sim, "T": torch.empty((case["nx"], case["ny"], case["nz"]), device=DEV),
            "out": {"T": torch.empty(n, device=DEV), "lheat": torch.empty(n, device=DEV)}}


def _prepare_adjoint(case, seed):
    sim, _, n, gen, _ = _sorted_sim(case, seed, adjoint_enabled=1, mc_enabled=0, heat_enabled=0, dt=2e-3)
    sim.levelset_update()
    sim.p2g()
    sim.extrapolate_bc(True)
    sim.synchronize()
    d = {"device": DEV, "dtype": torch.float64}
    st = {"sim": sim, "g_vel": torch.randn((n, 3), generator=gen, **d), "vel": torch.empty((n, 3), **d),
          "pos": torch.empty((n, 3), **d), "u": _face_set(case, torch.float64),
          "uold": _face_set(case, torch.float64), "ue": _face_set(case, torch.float64),
          "vel_p2g": torch.empty((n, 3), **d), "pos_p2g": torch.empty((n, 3), **d)}
    torch.cuda.synchronize()
    return st


def _prepare_step(case, seed):
    parts, n, gen, rng = _particles(case, seed)
    kw = dict(dt=1e-3, precision=case["precision"], rho_liquid=1000.0, tol=1e-6, refine_every=20, max_iters=20000,
              heat_enabled=1, heat_solver=mp.HEAT_JACOBI, heat_jacobi_iters=10, temperature0=1.0, mc_enabled=1,
              heat_alpha=[0.18, 0.08, 0.0, 0.0001, 0.08, 0.2], particle_capacity=n + n // 8 + 1024, seed=seed)
    if case["scene"] == "boiling":
        kw.update(rho_air=5.0, default_temperature=1.0, heat_add_bottom=1, heat_increase_bottom=0.2,
                  heat_bottom_clamp=1.2, heat_extend_boundary=1, heat_vacuum_neumann=1, melting_point=0.0,
                  boiling_point=1.05, liquid_heat_th=10.0, dissolve_gas_rate=0.95, gas_enabled=1, gas_every=2)
        t = (1.0, 0.01, 0.8, 10.0)
    else:
        kw.update(rho_air=1.0, solid_constraint=1, fix_solids=1, default_temperature=1.1, heat_add_bottom=0,
                  melting_point=1.0, boiling_point=10.0, liquid_heat_th=0.1, melt_enabled=1, freeze_enabled=1,
                  gas_enabled=0)
        t = (1.1, 0.0, 0.8, 0.1)
    cfg = _config(case, **kw)
    _attributes(parts, n, cfg, gen, *t)
    sim = mp.Simulator(cfg)
    if case["scene"] == "boiling":
        m = max(1, case["nx"] * case["ny"] // 256)
        x = rng.integers(3, [case["nx"] - 3, case["ny"] - 3], size=(m, 2))
        sim.set_seed_cells(np.unique((x[:, 0] * case["ny"] + x[:, 1]) * case["nz"] + 2))
    torch.cuda.synchronize()
    cells = (case["nx"], case["ny"], case["nz"])
    return {"sim": sim, "n": n, "in": parts, "out": _face_set(case),
            "cells": [torch.empty(cells, device=DEV) for _ in range(3)]}


def prepare(case, seed):
    st = globals()["_prepare_" + case["kind"]](case, seed)
    st["kind"] = case["kind"]
    return st


# ---- one pass ----
def _run_sort(s):
    mp.hash_sort_noalloc(s["cfg"], s["n"], s["pos"], *s["out"])
    return s["out"]


def _run_project(s):
    sim = s["sim"]
    for name, t in zip(FACES, s["in"]):
        _set(sim, name, t)
    sim.project()
    for name, t in zip(FACES, s["out"]):
        _get(sim, name, t)
    return s["out"]


def _run_transfer(s):
    sim = s["sim"]
    sim.p2g()
    sim.extrapolate_bc(True)
    sim.g2p()
    for name, t in zip(FACES, s["faces"]):
        _get(sim, name, t)
    _get_particles(sim, {"vel": s["vel"]})
    return s["faces"] + [s["vel"]]


def _run_surface(s):
    sim = s["sim"]
    sim.levelset_update()
    for name, t in zip(("LSFLUID", "LSAIR", "LSMERGE"), s["ls"]):
        _get(sim, name, t)
    _get(sim, "MARK", s["mark"])
    m = sim.marching_cubes()
    _check(sim, sim.L.mpf_get_mesh(sim.h, _ptr(s["verts"]), _ptr(s["tris"]), mp.DEVICE))
    _check(sim, sim.L.mpf_get_mesh_normals(sim.h, _ptr(s["normals"]), mp.DEVICE))
    return s["ls"] + [s["mark"], s["verts"], s["normals"], s["tris"], m["verts"], m["tris"]]


def _run_correct(s):
    sim = s["sim"]
    sim.set_particles(s["n"], where=mp.DEVICE, **s["in"])
    sim.hash_sort()
    sim.correct_positions()
    sim.hash_sort()
    _get_particles(sim, {"pos": s["pos"]})
    return s["pos"]


def _run_heat(s):
    sim = s["sim"]
    sim.heat()
    _get(sim, "TEMPERATURE", s["T"])
    _get_particles(sim, s["out"])
    return [s["T"], s["out"]["T"], s["out"]["lheat"]]


def _run_adjoint(s):
    sim, L, h = s["sim"], s["sim"].L, s["sim"].h
    u, uold, ue = _table(s["u"]), _table(s["uold"]), _table(s["ue"])
    _check(sim, L.mpf_g2p_adjoint(h, _ptr(s["g_vel"]), _ptr(s["vel"]), u, uold, _ptr(s["pos"]), mp.DEVICE))
    _check(sim, L.mpf_extrapolate_adjoint(h, u, ue, mp.DEVICE))
    _check(sim, L.mpf_p2g_adjoint(h, ue, _ptr(s["vel_p2g"]), _ptr(s["pos_p2g"]), mp.DEVICE))
    return [s["vel"], s["pos"], s["vel_p2g"], s["pos_p2g"]] + s["uold"] + s["ue"]


def _run_step(s):
    sim = s["sim"]
    sim.set_particles(s["n"], where=mp.DEVICE, **s["in"])
    sim.step(0)
    for name, t in zip(FACES + ["TEMPERATURE", "LSFLUID", "LSMERGE"], s["out"] + s["cells"]):
        _get(sim, name, t)
    return s["out"] + s["cells"]


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---- what a pass cannot do without ----
def work(case):
    """Bytes: inputs read once, outputs written once (per cell, per face set, per particle). Flops are the few
    per element that each stage's formulas need."""
    G = case["nx"] * case["ny"] * case["nz"]
    P = 8 * G * case["fill"]
    faces = 6 * 4 * G
    k = case["kind"]
    if k == "sort":
        return {"bytes": P * (12 + 8) + 8 * G, "flops": 6 * P}
    if k == "project":  # velocities in and out, cell types and level set
        return {"bytes": 2 * faces + 5 * G, "flops": 30 * G}
    if k == "transfer":  # position, velocity, mass, type; faces and snapshot; velocity out
        return {"bytes": P * (12 + 12 + 4 + 1 + 12) + 2 * faces + 21 * G, "flops": 54 * 12 * P}
    if k == "surface":
        return {"bytes": P * 13 + 8 * G + 13 * G, "flops": 60 * G}
    if k == "correct":  # the particle record in and out once per sort, positions through the correction
        return {"bytes": P * (4 * 45 + 25) + 16 * G, "flops": 64 * 8 * P}
    if k == "heat":
        return {"bytes": P * (12 + 1 + 8 + 8) + 20 * G, "flops": 27 * 12 * P}
    if k == "adjoint":
        return {"bytes": P * (12 + 12 + 1 + 5 * 24) + 4 * 2 * faces, "flops": 2 * 54 * 20 * P}
    return {"bytes": P * (8 * 45 + 100) + 6 * faces + 60 * G, "flops": 54 * 40 * P}


# ---- 64-bit values ----
def _pad(t, value):
    return torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1), value=value)


def _exact_project(case, seed):
    """Divergence, Jacobi-preconditioned CG to 1e-13 and the pressure gradient in FP64."""
    mark, ls, faces = _faces_and_marks(case, seed)
    faces = [f.double() for f in faces]
    h = float(np.float32(H))
    solid_c = case["solids"] > 0
    il, ia = 1.0 / 1000.0, 1.0 / case["rho_air"]
    n = [case["nx"], case["ny"], case["nz"]]
    M, LS = _pad(mark.float(), float(mp.TYPEBOUNDARY)).to(torch.int8), _pad(ls.double(), 0.0)

    def pair(t, a):  # the cells below and above every face of axis a
        lo = [slice(1, -1)] * 3
        hi = [slice(1, -1)] * 3
        lo[a], hi[a] = slice(0, -1), slice(1, None)
        return t[tuple(lo)], t[tuple(hi)]

    beta, cell_flux = [], []
    for a in range(3):
        ml, mh = pair(M, a)
        ll, lh = pair(LS, a)
        ul, uh = (ml == 0) | (ml == 1), (mh == 0) | (mh == 1)
        closed = (ml == mp.TYPEBOUNDARY) | (mh == mp.TYPEBOUNDARY)
        sol = (ml == mp.TYPESOLID) | (mh == mp.TYPESOLID)
        if solid_c:
            closed = closed | sol
        mixed = ul & uh & (ml != mh)
        th = torch.where(mixed, -ll / torch.where(mixed, lh - ll, 1.0), 0.0)
        bl = torch.where(ml == 0, il, ia)
        bh = torch.where(mh == 0, il, ia)
        b = torch.where(mixed, bh + th.clamp(0, 1) * (bl - bh), torch.where(ul, bl, bh))
        beta.append(torch.where(closed | ~(ul | uh), 0.0, b))
        w, r = faces[a], faces[a + 3]
        # the velocity each side's cell sees: its own phase's, or both blended across a liquid/air face
        own_l, oth_l = torch.where(ml == 0, w, r), torch.where(ml == 0, r, w)
        own_h, oth_h = torch.where(mh == 0, w, r), torch.where(mh == 0, r, w)
        vl = torch.where(mixed, th * own_l + (1 - th) * oth_l, own_l)
        thh = torch.where(mixed, -lh / torch.where(mixed, ll - lh, 1.0), 0.0)
        vh = torch.where(mixed, thh * own_h + (1 - thh) * oth_h, own_h)
        if solid_c:
            vl, vh = torch.where(mh == mp.TYPESOLID, 0.0, vl), torch.where(ml == mp.TYPESOLID, 0.0, vh)
        cell_flux.append((vl.narrow(a, 1, n[a]), vh.narrow(a, 0, n[a])))
    unk = (mark == 0) | (mark == 1)
    rhs = sum(hi - lo for hi, lo in cell_flux) / h
    rhs = torch.where(unk, rhs, 0.0)
    del cell_flux

    diag = sum(beta[a].narrow(a, 0, n[a]) + beta[a].narrow(a, 1, n[a]) for a in range(3))
    dinv = torch.where(unk & (diag > 0), -h * h / torch.where(diag > 0, diag, 1.0), 0.0)

    def apply(p):
        out = None
        for a in range(3):
            lo, hi = n[a] - 1, 1
            f = beta[a].narrow(a, 1, n[a] - 1) * (p.narrow(a, 1, n[a] - 1) - p.narrow(a, 0, n[a] - 1))
            if out is None:
                out = torch.zeros_like(p)
            out.narrow(a, 0, lo).add_(f)
            out.narrow(a, hi, lo).sub_(f)
        return torch.where(unk, out, 0.0).div_(h * h)

    x = torch.zeros_like(rhs)
    r = rhs.clone()
    z = r * dinv
    p = z.clone()
    rz = torch.sum(r * z)
    stop = 1e-13 * float(torch.linalg.vector_norm(rhs))
    for it in range(20000):
        q = apply(p)
        al = rz / torch.sum(p * q)
        x += al * p
        r -= al * q
        if it % 50 == 49 and float(torch.linalg.vector_norm(r)) <= stop:
            break
        z = r * dinv
        new = torch.sum(r * z)
        p.mul_(new / rz).add_(z)
        rz = new
    out = []
    for f in range(6):
        a, w = f % 3, il if f < 3 else ia
        u = faces[f].clone()
        g = (x.narrow(a, 1, n[a] - 1) - x.narrow(a, 0, n[a] - 1)) / h
        inner = u.narrow(a, 1, n[a] - 1)
        inner -= w * g
        if solid_c:
            s = mark == mp.TYPESOLID
            inner.masked_fill_(s.narrow(a, 1, n[a] - 1) | s.narrow(a, 0, n[a] - 1), 0.0)
        out.append(u)
    return out


def exact(case, seed):
    if case["kind"] != "project":
        return None
    return _exact_project(case, seed)

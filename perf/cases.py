"""The work whose time is watched: what programs on this library have it do,
through the entry points that they call (flip2_amd and the C ABI of
include/flip2.h), from the smallest calls to the largest configuration.

Sorting, scanning and the particle-to-grid transfer take device arrays.  The
FLIP simulation (FluidSim) keeps its particles on the device and advances them
at every pass, as a program's frame loop does; its velocity field is read back
into pinned memory after the step (the pressure where the grid is too large to
read back at every step).  The host-driven frame, the U-Net gradient and the
reference-compatible frame take host arrays, as those entry points do.
"""
from __future__ import annotations

import ctypes
import math
import os

import numpy as np
import torch

import flip2_amd as F

ROOT = F.REPO_ROOT
NET = os.path.join(ROOT, "flip2_amd", "data", "c4_unet_16_32_64.npy")
GRAVITY, FLIP, MARGIN = -9.81, 0.95, 1e-3
RC_DT = 1.0 / 240.0
PPC = 8  # particles per fluid cell (jittered 2 x 2 x 2)


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # key/value sort of a small list: a few nodes' worth of keys, where launches are all of the time
        dict(name="sort_small", kind="sort", n=4099, begin=0, end=32, values=True, bits=32),
        # the microbench of the largest transfer: 24-bit cell keys of 2^24 particles, sorted to a permutation
        dict(name="sort_large", kind="sort", n=16777259, begin=0, end=24, values=False, bits=24),
        # transfer of a small cloud from separate arrays (what transfer() and small tools call)
        dict(name="transfer_small", kind="transfer", n=20000, nx=32, ny=32, nz=32, records=False, order="shuffled"),
        # transfer microbench: 2^24 particles, 256^3, fully shuffled records
        dict(name="transfer_large", kind="transfer", n=16777216, nx=256, ny=256, nz=256, records=True, order="shuffled"),
        # a frame driven from host arrays (an add-on or a notebook): particles in, one step, particles out
        dict(name="host_frame_24", kind="host", nx=24, ny=16, nz=24, scene="dam", prec="jacobi"),
        # the plain dam break, 64^3, 503k particles, Jacobi-PCG
        dict(name="step_dam_64", kind="step", nx=64, ny=64, nz=64, scene="dam", prec="jacobi", dt=1.0 / 240.0),
        # a wave tank on an uneven grid, MIC(0)-PCG: most of the domain is fluid
        dict(name="step_tank_mic", kind="step", nx=168, ny=104, nz=136, scene="tank", prec="mic0", dt=1.0 / 240.0),
        # colliding spheres, 512^3 in 8^3 bricks, 30M particles, MIC(0)-PCG: the largest configuration; the time
        # step moves a particle one cell
        dict(name="step_spheres_512", kind="step", nx=512, ny=512, nz=512, scene="spheres", prec="mic0", dt=1.0 / 1024.0),
        # adaptive time steps with a static obstacle and a moving paddle: two CFL-limited substeps per frame
        dict(name="frame_paddle_96", kind="frame", nx=128, ny=72, nz=96, scene="tank", prec="mic0", frame=1.0 / 60.0),
        # pressure solve with the learned preconditioner: the 128^3 dam break with a sphere, committed network
        dict(name="solve_learned_128", kind="learned", n=128),
        # one training step's forward and backward pass of the network
        dict(name="unet_grad_64", kind="grad", n=64),
        # one substep of the reference-compatible path, FP64, stage by stage: the smoke scene's block on a 32^3
        # grid (its own frame loop takes any number of substeps and solver retries, by the particles' velocities)
        dict(name="rc_substep_32", kind="rc", n=32, bx=12, by=16, bz=32, sweeps=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _eight(rng, lo, hi):
    return 8 * max(1, _log(rng, lo, hi) // 8)


def draw(rng):
    kind = rng.choice(["sort", "sort", "scan", "transfer", "transfer", "host", "step", "step", "step", "frame", "learned", "grad", "rc"])
    if kind == "sort":
        end = rng.choice([8, 15, 18, 21, 24, 27, 32])
        return dict(kind=kind, n=_log(rng, 100, 1.6e7) | 1, begin=0, end=end, values=rng.random() < 0.5, bits=rng.choice([end, 32]))
    if kind == "scan":
        return dict(kind=kind, n=_log(rng, 1000, 1.6e7) | 1, exclusive=rng.random() < 0.5, high=rng.choice([2, 64, 1 << 31]))
    if kind == "transfer":
        n = _log(rng, 1000, 1.2e7) | 1
        side = max(16, min(248, int(round((n / rng.choice([1, 2, 8])) ** (1 / 3) / 8)) * 8))
        return dict(kind=kind, n=n, nx=side, ny=_eight(rng, max(8, side // 2), side), nz=side, records=rng.random() < 0.5, order=rng.choice(["shuffled", "cells"]))
    if kind == "host":
        return dict(kind=kind, nx=_eight(rng, 16, 48), ny=_eight(rng, 16, 48), nz=_eight(rng, 16, 40), scene=rng.choice(["dam", "tank"]), prec=rng.choice(["jacobi", "mic0"]))
    if kind == "step":
        scene = rng.choice(["dam", "tank", "spheres"])
        hi = 320 if scene == "spheres" else 176
        return dict(kind=kind, nx=_eight(rng, 32, hi), ny=_eight(rng, 32, hi * 2 // 3), nz=_eight(rng, 32, hi), scene=scene, prec=rng.choice(["jacobi", "mic0", "mic0"]), dt=round(1.0 / rng.uniform(240, 480), 6))
    if kind == "frame":
        return dict(kind=kind, nx=_eight(rng, 64, 144), ny=_eight(rng, 48, 96), nz=_eight(rng, 32, 112), scene="tank", prec=rng.choice(["jacobi", "mic0"]), frame=1.0 / 60.0)
    if kind == "learned":
        return dict(kind=kind, n=_eight(rng, 48, 128))
    if kind == "grad":
        return dict(kind=kind, n=_eight(rng, 24, 88))
    n = rng.randint(12, 40)
    return dict(kind=kind, n=n, bx=rng.randint(4, n // 2), by=rng.randint(4, n // 2), bz=rng.randint(5, n), sweeps=rng.choice([16, 64, 200]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _grid(case):
    return (0.0, 0.0, 0.0, case["nx"], case["ny"], case["nz"], 1.0 / max(case["nx"], case["ny"], case["nz"]))


def _flow(x, y, z, rng, amp=0.6, modes=3):
    """A smooth seeded velocity field at the given positions."""
    out = []
    for _ in range(3):
        v = torch.zeros_like(x)
        for _ in range(modes):
            f = rng.integers(1, 5, 3)
            a, ph = rng.uniform(-amp, amp), rng.uniform(0, 2 * math.pi)
            v += a / math.sqrt(modes) * torch.sin(2 * math.pi * (f[0] * x + f[1] * y + f[2] * z) + ph)
        out.append(v)
    return out


def _jitter(cells, nx, ny, h, gen):
    """PPC jittered particles in each of the given cells (x fastest)."""
    sub = torch.arange(PPC, device="cuda").repeat(cells.numel())
    c = cells.repeat_interleave(PPC)
    u = torch.rand(3, c.numel(), device="cuda", generator=gen, dtype=torch.float32)
    i, j, k = c % nx, (c // nx) % ny, c // (nx * ny)
    return [(i_.float() + ((sub >> s & 1).float() + u[s]) * 0.5) * h for s, i_ in enumerate((i, j, k))]


def _scene(case, seed, sphere=False):
    """(x, y, z, vx, vy, vz) of a scene on the device; with `sphere`, none inside the static sphere (see _sphere)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = _grid(case)[6]
    gen, rng = _gen(seed), np.random.default_rng(seed)
    lx, ly = nx * h, ny * h

    def axis(n):
        return (torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) * h

    X, Y, Z = axis(nx)[None, None, :], axis(ny)[None, :, None], axis(nz)[:, None, None]
    phase = [float(v) for v in rng.uniform(0, 2 * math.pi, 3)]
    if case["scene"] == "dam":
        mask = (X < 0.4 * lx + h) & (Y < 0.6 * ly + h) & (Z > -1)
    elif case["scene"] == "tank":
        mask = (Y < 0.56 * ly + h) & (X > -1) & (Z > -1)
    else:
        m = min(nx, ny, nz) * h
        r = 0.15 * (m if nx == ny == nz else 1.6 * m)
        centres = [(0.5 * lx + s * (r + 0.002), 0.5 * ly, 0.5 * nz * h) for s in (-1.0, 1.0)]
        mask = torch.zeros(nz, ny, nx, dtype=torch.bool, device="cuda")
        for c in centres:
            mask |= (X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2 <= (r + h) ** 2
    cells = torch.nonzero(mask.reshape(-1)).reshape(-1)
    x, y, z = _jitter(cells, nx, ny, h, gen)
    if case["kind"] == "host":  # whole cells: as many particles for every seed
        keep = torch.ones_like(x, dtype=torch.bool)
    elif case["scene"] == "dam":
        keep = (x < 0.4 * lx) & (y < 0.6 * ly)
    elif case["scene"] == "tank":
        keep = y < 0.5 * ly + 0.02 * ly * (torch.sin(6.0 * x + phase[0]) + torch.sin(9.0 * z + phase[1]) * torch.sin(4.0 * x + phase[2]))
        keep &= x >= 0.06
    else:
        keep = torch.zeros_like(x, dtype=torch.bool)
        for c in centres:
            keep |= (x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2 <= r * r
    if sphere:
        c, rs = _sphere(case)
        keep &= (x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2 > rs * rs
    x, y, z = x[keep], y[keep], z[keep]
    v = _flow(x, y, z, rng)
    if case["scene"] == "spheres":
        v[0] += torch.where(x < 0.5 * lx, 2.0, -2.0)
    return [x, y, z] + v


def _sphere(case):
    h = _grid(case)[6]
    return (0.6 * case["nx"] * h, 0.2 * case["ny"] * h + 0.05, 0.5 * case["nz"] * h), 0.1


def _solid(case):
    """Static solid sphere: bytes [z][y][x]."""
    h = _grid(case)[6]
    c, r = _sphere(case)
    z, y, x = (((np.arange(case[k]) + 0.5) * h) for k in ("nz", "ny", "nx"))
    d = (x[None, None, :] - c[0]) ** 2 + (y[None, :, None] - c[1]) ** 2 + (z[:, None, None] - c[2]) ** 2
    return (d <= r * r).astype(np.uint8)


def _paddle(t):
    """The paddle's face and velocity at time t."""
    w = 2 * math.pi
    return 0.03 + 0.02 * math.sin(w * t), 0.02 * w * math.cos(w * t)


def _sim(case, parts, **more):
    sim = F.FluidSim(parts[0].numel(), _grid(case), gravity=GRAVITY, flip=FLIP, margin=MARGIN, **more)
    host = [p.cpu().numpy() for p in parts]
    sim.set_particles(*host)
    return sim, host


class _Device:
    """A torch tensor where the package takes one of its device buffers."""

    def __init__(self, t):
        self.ptr = t.data_ptr()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sort":
        n, gen = case["n"], _gen(seed)
        keys = torch.randint(0, 1 << case["bits"], (n,), device="cuda", generator=gen, dtype=torch.int64).to(torch.int32) if case["bits"] < 32 else \
            torch.randint(-(1 << 31), 1 << 31, (n,), device="cuda", generator=gen, dtype=torch.int64).to(torch.int32)
        vals = torch.randint(0, 1 << 30, (n,), device="cuda", generator=gen, dtype=torch.int32) if case["values"] else None
        ws = F.lib().flip2_sort_workspace_bytes(n, case["begin"], case["end"])
        return dict(case=case, keys=keys, vals=vals, out=[torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(4)],
                    ws=torch.empty(ws, dtype=torch.uint8, device="cuda"))
    if kind == "scan":
        n = case["n"]
        v = torch.randint(0, case["high"], (n,), device="cuda", generator=_gen(seed), dtype=torch.int64).to(torch.int32)
        ws = F.lib().flip2_scan_workspace_bytes(n)
        return dict(case=case, v=v, out=torch.empty_like(v), total=torch.empty(1, dtype=torch.int32, device="cuda"),
                    ws=torch.empty(ws, dtype=torch.uint8, device="cuda"))
    if kind == "transfer":
        parts = _cloud(case, seed)
        cells = case["nx"] * case["ny"] * case["nz"]
        if case["records"]:
            rec = torch.zeros(case["n"], 8, device="cuda")
            for c, p in enumerate(parts):
                rec[:, c] = p
            parts = [rec]
        return dict(case=case, parts=parts, pipe=F.P2GPipeline(case["n"], _grid(case)), out=[torch.empty(cells, device="cuda") for _ in range(3)])
    if kind in ("step", "frame"):
        frame = kind == "frame"
        parts = _scene(case, seed, sphere=frame)
        sim, _ = _sim(case, parts, preconditioner=case["prec"], dt=case.get("dt", 1.0 / 240.0))
        if frame:
            sim.set_solid(_solid(case))
        cells = case["nx"] * case["ny"] * case["nz"]
        state = dict(case=case, sim=sim, t=0.0)
        if _fields(case):
            state["pinned"] = [torch.empty(cells, pin_memory=True) for _ in range(3)]
        else:  # p: 512 doubles per active brick, one brick in sixteen at most; 0 past the last
            state["pinned"] = [torch.zeros(cells // 16, dtype=torch.float64, pin_memory=True)]
        return state
    if kind == "host":
        sim, host = _sim(case, _scene(case, seed), preconditioner=case["prec"])
        return dict(case=case, sim=sim, host=host)
    if kind == "learned":
        c = _learned_scene(case)
        parts = _scene(c, seed, sphere=True)
        sim, _ = _sim(c, parts, preconditioner="learned")
        sim.set_solid(_solid(c))
        net = F.UNet(case["n"])
        net.set_params(np.load(NET, allow_pickle=False))
        sim.set_unet(net)
        for s in ("transfer", "prepare", "system"):
            sim.stage(s)
        return dict(case=case, sim=sim, net=net, pinned=[torch.empty(case["n"] ** 3, dtype=torch.float64, pin_memory=True)])
    if kind == "grad":
        b, coef = _dense_system(case, seed)
        net = F.UNet(case["n"])
        net.set_params(np.load(NET, allow_pickle=False))
        return dict(case=case, net=net, b=b.float().cpu().numpy(), coef=coef.cpu().numpy().astype(np.uint16))
    pos, vel = _block(case, seed)
    p = F.Particles(pos[0].size)
    n = case["n"]
    p.setDomain(0.0, 0.0, 0.0, n, n, n, 1.0 / n)
    return dict(case=case, p=p, pos=pos, vel=vel)


def _fields(case):
    """Whether the velocity field is small enough to be read back at every step."""
    return case["nx"] * case["ny"] * case["nz"] <= 1 << 24


def _cloud(case, seed):
    """Particles uniform in the grid, velocities uniform in [-1, 1); "cells": in the order of their cells, slightly moved, as a step leaves them."""
    gen, n, h = _gen(seed), case["n"], _grid(case)[6]
    u = torch.rand(6, n, device="cuda", generator=gen, dtype=torch.float32)
    p = [u[d] * (case[k] * h) for d, k in enumerate(("nx", "ny", "nz"))]
    if case["order"] == "cells":
        c = [torch.floor(a / h).long().clamp(0, case[k] - 1) for a, k in zip(p, ("nx", "ny", "nz"))]
        nb = [case[k] // 8 for k in ("nx", "ny", "nz")]
        key = (((c[2] >> 3) * nb[1] + (c[1] >> 3)) * nb[0] + (c[0] >> 3)) * 512 + (c[2] & 7) * 64 + (c[1] & 7) * 8 + (c[0] & 7)
        order = torch.argsort(key)
        move = (torch.rand(3, n, device="cuda", generator=gen, dtype=torch.float32) - 0.5) * h
        p = [(a[order] + move[d]).clamp(0, case[k] * h * 0.999999) for d, (a, k) in enumerate(zip(p, ("nx", "ny", "nz")))]
    return p + [u[d] * 2 - 1 for d in (3, 4, 5)]


def _learned_scene(case):
    return dict(kind="learned", nx=case["n"], ny=case["n"], nz=case["n"], scene="dam")


def _dense_system(case, seed):
    """A residual and operator on a dense n^3 grid, float64 and int64 [z][y][x]: fluid in a block whose surface is uneven."""
    n, rng, gen = case["n"], np.random.default_rng(seed), _gen(seed)
    a = (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) / n
    X, Y, Z = a[None, None, :], a[None, :, None], a[:, None, None]
    ph = [float(v) for v in rng.uniform(0, 6.28, 3)]
    fluid = Y < 0.35 + 0.08 * torch.sin(6 * X + ph[0]) + 0.08 * torch.sin(7 * Z + ph[1]) * torch.sin(5 * X + ph[2])
    coef = _coefficients(fluid, torch.zeros_like(fluid))
    x, y, z = torch.broadcast_tensors(X, Y, Z)
    b = sum(_flow(x, y, z, rng, amp=1.0, modes=4)) + 0.3 * torch.randn(n, n, n, device="cuda", generator=gen, dtype=torch.float64)
    return (b * fluid).float().double(), coef


def _block(case, seed):
    """A block of jittered particles with random velocities, FP64 host arrays."""
    n, gen = case["n"], _gen(seed)
    k, j, i = torch.meshgrid(torch.arange(case["bz"]), torch.arange(case["by"]), torch.arange(case["bx"]), indexing="ij")
    cells = (i + 2 + n * j + n * n * k).reshape(-1).cuda()
    pos = [a.double().cpu().numpy() for a in _jitter(cells, n, n, 1.0 / n, gen)]
    v = torch.rand(3, pos[0].size, device="cuda", generator=gen, dtype=torch.float32) - 0.5
    return pos, [a.double().cpu().numpy() for a in v]


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _read(sim, name, buf):
    """An array of the simulation into pinned memory (flip2_fluid_get_array)."""
    count = ctypes.c_size_t()
    F.check(F.lib().flip2_fluid_get_array(sim._h, name, buf.data_ptr(), buf.numel(), ctypes.byref(count)))
    return buf[:count.value]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "sort":
        o = s["out"]
        F.check(F.lib().flip2_sort_pairs_u32(s["keys"].data_ptr(), s["vals"].data_ptr() if s["vals"] is not None else None, *(t.data_ptr() for t in o),
                                             case["n"], case["begin"], case["end"], s["ws"].data_ptr(), s["ws"].numel(), _stream()))
        return o[:2]
    if kind == "scan":
        F.check(F.lib().flip2_scan_u32(s["v"].data_ptr(), s["out"].data_ptr(), case["n"], int(case["exclusive"]), s["total"].data_ptr(),
                                       s["ws"].data_ptr(), s["ws"].numel(), _stream()))
        return s["out"], s["total"]
    if kind == "transfer":
        out = [_Device(t) for t in s["out"]]
        if case["records"]:
            s["pipe"].run_records(case["n"], _Device(s["parts"][0]), out, _stream())
        else:
            s["pipe"].run(case["n"], [_Device(t) for t in s["parts"]], out, _stream())
        return s["out"]
    if kind == "step":
        s["sim"].step()
        if _fields(case):
            return [_read(s["sim"], name, buf) for name, buf in zip((b"U", b"V", b"W"), s["pinned"])]
        _read(s["sim"], b"p", s["pinned"][0])
        return s["pinned"][0]
    if kind == "frame":
        face, speed = _paddle(s["t"])
        s["sim"].set_solid_box((0.0, 0.0, 0.0), (face, 10.0, 10.0), (speed, 0.0, 0.0))
        s["sim"].step_frame(case["frame"], cfl=0.5, max_substeps=2)
        s["t"] += case["frame"]
        return [_read(s["sim"], name, buf) for name, buf in zip((b"U", b"V", b"W"), s["pinned"])]
    if kind == "host":
        s["sim"].set_particles(*s["host"])
        s["sim"].step()
        return s["sim"].particles()
    if kind == "learned":
        s["sim"].solve_with("learned")
        return _read(s["sim"], b"p", s["pinned"][0])
    if kind == "grad":
        return s["net"].loss_grad(s["b"], s["coef"])
    p = s["p"]
    p.set_positions(*s["pos"])
    p.set_velocities(*s["vel"])
    p.setTime(RC_DT, RC_DT)
    p.initialize()
    p.particleVelToVoxels()
    p.applyGravity(RC_DT)
    p.calcDivU()
    p.gsIterations(RC_DT, case["sweeps"])
    p.updateVoxelVelocities()
    p.voxelVelsToParticles()
    p.advectParticles()
    p.moveSolidParticles()
    return p.positions(), p.velocities()


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _count(case):
    """Particles of a scene, about."""
    cells = case["nx"] * case["ny"] * case["nz"]
    if case["scene"] == "spheres":
        m = min(case["nx"], case["ny"], case["nz"])
        r = 0.15 * (m if case["nx"] == case["ny"] == case["nz"] else 1.6 * m)
        return PPC * 2 * 4.19 * r ** 3
    return PPC * cells * (0.24 if case["scene"] == "dam" else 0.5)


def work(case):
    kind = case["kind"]
    if kind == "sort":
        return {"bytes": case["n"] * (16 if case["values"] else 12), "flops": 0}
    if kind == "scan":
        return {"bytes": 8 * case["n"], "flops": 0}
    if kind == "transfer":
        return {"bytes": 24 * case["n"] + 12 * case["nx"] * case["ny"] * case["nz"], "flops": 24 * 6 * case["n"]}
    if kind in ("step", "frame", "host"):
        # the particles in and out, and the fluid's faces (six fields); of the solve, the system in and the
        # pressure out: no number of iterations is taken as given
        n = _count(case) * (2 if kind == "frame" else 1)
        return {"bytes": 48 * n + (48 + 18) * n / PPC, "flops": 600 * n}
    if kind == "learned":
        cells = 0.24 * case["n"] ** 3
        return {"bytes": 18 * cells, "flops": 2 * 27 * cells * (2 * 16 * 16 + 48 * 16 + 16 * 16)}
    if kind == "grad":
        n = case["n"]
        conv = 2 * 27 * (n ** 3 * (2 * 16 + 16 * 16 + 48 * 16 + 16 * 16) + (n // 2) ** 3 * (16 * 32 + 2 * 32 * 32 + 96 * 32) + (n // 4) ** 3 * (32 * 64 + 64 * 64))
        return {"bytes": 6 * n ** 3 + 4 * 2 * 290000, "flops": 3 * conv}
    n = PPC * case["bx"] * case["by"] * case["bz"]
    return {"bytes": 96 * n, "flops": 2 * 64 * 3 * 20 * n + 20 * case["sweeps"] * 100 * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sort", "scan"):
        return "exact"
    if kind == "transfer":
        return {"rel": 1e-6, "max": 1e-4}  # FP32 results of sums held in 64 bits: 4e-8 off
    if kind == "frame":
        # between the substeps positions are rounded to FP32: a particle on the other side of a cell's face makes
        # that cell fluid or air (8e-4 from the exact fields where one does, 3e-7 where none does)
        return {"rel": 3e-3, "max": 0.99}
    if kind == "step":
        # the solver stops at a relative residual of 1e-6: Jacobi's and MIC(0)'s fields are 1e-7 to 3e-7 apart,
        # single faces 3e-5, pressures 9e-7
        return {"rel": 4e-6, "max": 3e-4}
    if kind == "host":
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "learned":
        return {"rel": 1e-5, "max": 3e-4}  # pressures: 6e-7 to 2e-6 from the exact ones
    if kind == "grad":
        return {"rel": 1e-2, "max": 0.3}  # BF16 weights, activations and gradients: 1e-2 from the exact ones
    return {"rel": 1e-9, "max": 1e-6}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_AX = (2, 1, 0)  # tensor dimension of axis x, y, z in [z][y][x]


def _shift(a, axis, step, fill=0):
    """b[c] = a[c + step along axis], `fill` outside."""
    d = _AX[axis]
    b = torch.full_like(a, fill)
    n = a.shape[d]
    if step > 0:
        b.narrow(d, 0, n - 1).copy_(a.narrow(d, 1, n - 1))
    else:
        b.narrow(d, 1, n - 1).copy_(a.narrow(d, 0, n - 1))
    return b


def _coefficients(fluid, solid):
    """diag | fluid-neighbour mask << 3 of the fluid cells; outside the grid is solid."""
    diag, mask = torch.zeros_like(fluid, dtype=torch.int64), torch.zeros_like(fluid, dtype=torch.int64)
    for d in range(6):
        step = 1 if d & 1 else -1
        diag += (~_shift(solid, d >> 1, step, True)).long()
        mask |= _shift(fluid, d >> 1, step, False).long() << d
    return torch.where(fluid, diag | mask << 3, torch.zeros_like(diag))


def _operator(coef):
    diag = (coef & 7).double()
    on = [((coef >> 3 >> d) & 1).double() for d in range(6)]

    def apply(x):
        y = diag * x
        for d in range(6):
            y -= on[d] * _shift(x, d >> 1, 1 if d & 1 else -1)
        return y

    return apply, diag


def _cg(coef, b, tol=1e-13, most=6000):
    apply, diag = _operator(coef)
    inv = torch.where(diag > 0, 1.0 / diag.clamp(min=1), torch.zeros_like(diag))
    x, r = torch.zeros_like(b), b.clone()
    p = z = inv * r
    rz, stop = (r * z).sum(), tol * b.norm()
    for it in range(most):
        q = apply(p)
        alpha = rz / (p * q).sum()
        x = x + alpha * p
        r = r - alpha * q
        if it % 16 == 0 and r.norm() <= stop:
            break
        z = inv * r
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def _weights(q, axis, size):
    """Per dimension: the two nodes below and above, and their weights, for a component normal to `axis`."""
    out = []
    for d in range(3):
        v = q[d] if d == axis else q[d] - 0.5
        f = torch.floor(v)
        t = v - f
        i = f.long()
        out.append([(i, 1 - t, (i >= 0) & (i < size[d])), (i + 1, t, (i + 1 >= 0) & (i + 1 < size[d]))])
    return out


def _corners(q, axis, size):
    w = _weights(q, axis, size)
    for x, wx, ox in w[0]:
        for y, wy, oy in w[1]:
            for z, wz, oz in w[2]:
                ok = ox & oy & oz
                yield torch.where(ok, x + size[0] * (y + size[1] * z), torch.zeros_like(x)), torch.where(ok, wx * wy * wz, torch.zeros_like(wx))


def _splat(q, v, axis, size):
    n = size[0] * size[1] * size[2]
    m, w = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.zeros(n, dtype=torch.float64, device="cuda")
    for idx, wt in _corners(q, axis, size):
        m.index_add_(0, idx, wt * v)
        w.index_add_(0, idx, wt)
    return torch.where(w > 0, m / torch.where(w > 0, w, torch.ones_like(w)), torch.zeros_like(m)).reshape(size[2], size[1], size[0])


def _sample(f, q, axis, size):
    out = torch.zeros_like(q[0])
    for idx, wt in _corners(q, axis, size):
        out += wt * f.reshape(-1)[idx]
    return out


def _tiled(a):
    nz, ny, nx = a.shape
    return a.reshape(nz // 8, 8, ny // 8, 8, nx // 8, 8).permute(0, 2, 4, 1, 3, 5).reshape(-1)


def _f32(v):
    return float(np.float32(v))


class _Flip64:
    """The FLIP step on dense FP64 fields."""

    def __init__(self, case, parts, static=None):
        self.size = [case["nx"], case["ny"], case["nz"]]
        self.h = _f32(_grid(case)[6])
        self.x = [p.double() for p in parts[:3]]
        self.v = [p.double() for p in parts[3:]]
        shape = (case["nz"], case["ny"], case["nx"])
        self.static = torch.zeros(shape, dtype=torch.bool, device="cuda") if static is None else torch.from_numpy(static).cuda().bool()
        self.box = None

    def set_box(self, face, speed):
        self.box = (_f32(face), _f32(speed))
        xc = (torch.arange(self.size[0], device="cuda", dtype=torch.float64) + 0.5) * self.h
        self.inbox = (xc < self.box[0])[None, None, :].expand(self.static.shape)

    def transfer(self):
        self.q = [x / self.h for x in self.x]
        self.F = [_splat(self.q, self.v[a], a, self.size) for a in range(3)]

    def system(self, dt):
        dt = _f32(dt)
        solid = self.static | self.inbox if self.box else self.static
        self.solid = solid
        self.F0 = []
        for a in range(3):
            below = _shift(solid, a, -1, True)
            wall = solid | below
            speed = torch.zeros_like(self.F[a])
            if self.box and a == 0:
                edge = torch.ones_like(solid)
                edge.narrow(_AX[a], 0, 1).fill_(False)
                speed = torch.where(edge & (self.inbox | _shift(self.inbox, a, -1, False)), self.box[1], 0.0)
            f = torch.where(wall, speed, self.F[a])
            self.F0.append(f)
            self.F[a] = torch.where(wall, f, f + _f32(np.float32(GRAVITY) * np.float32(dt))) if a == 1 else f.clone()
        c = [torch.floor(q).long().clamp(0, n - 1) for q, n in zip(self.q, self.size)]
        count = torch.bincount(c[0] + self.size[0] * (c[1] + self.size[1] * c[2]), minlength=solid.numel()).reshape(solid.shape)
        self.fluid = (count > 0) & ~solid
        self.coef = _coefficients(self.fluid, solid)
        div = sum(_shift(self.F[a], a, 1) - self.F[a] for a in range(3))
        self.b = torch.where(self.fluid, -(self.h / dt) * div, torch.zeros_like(div))

    def solve(self):
        self.p = _cg(self.coef, self.b)

    def project(self, dt):
        s = _f32(np.float32(dt) / np.float32(self.h))
        for a in range(3):
            below = _shift(self.solid, a, -1, True)
            on = ~self.solid & ~below & (self.fluid | _shift(self.fluid, a, -1, False))
            self.F[a] = torch.where(on, self.F[a] - s * (self.p - _shift(self.p, a, -1)), self.F[a])

    def move(self, dt):
        dt, m = _f32(dt), _f32(np.float32(MARGIN) * np.float32(self.h))
        flip = _f32(FLIP)
        pic = [_sample(self.F[a], self.q, a, self.size) for a in range(3)]
        old = [_sample(self.F0[a], self.q, a, self.size) for a in range(3)]
        self.v = [flip * (v + n - o) + (1 - flip) * n for v, n, o in zip(self.v, pic, old)]
        mid = [(x + 0.5 * dt * u) / self.h for x, u in zip(self.x, pic)]
        new = [x + dt * _sample(self.F[a], mid, a, self.size) for a, x in enumerate(self.x)]
        new = [x.clamp(m, n * self.h - m) for x, n in zip(new, self.size)]
        if self.box:  # out of the paddle through its face
            new[0] = torch.where(new[0] < self.box[0], torch.full_like(new[0], self.box[0] + m), new[0])
        c = [torch.floor(x / self.h).long().clamp(0, n - 1) for x, n in zip(new, self.size)]
        idx = c[0] + self.size[0] * (c[1] + self.size[1] * c[2])
        stuck = self.solid.reshape(-1)[idx]
        if self.box:
            stuck &= ~self.inbox.reshape(-1)[idx]
        self.x = [torch.where(stuck, a, b) for a, b in zip(self.x, new)]

    def step(self, dt):
        self.system(dt)
        self.solve()
        self.project(dt)


def _slots(p, fluid):
    """A cell field in the solver's order: the bricks with fluid, 512 cells each."""
    active = _tiled(fluid.long()).reshape(-1, 512).any(dim=1)
    return _tiled(p).reshape(-1, 512)[active].reshape(-1)


def _conv(x, w, bias):
    """3 x 3 x 3 correlation, zero padding: x [n, n, n, cin], w [27, cout, cin]."""
    n = x.shape[0]
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    y = bias.expand(n, n, n, -1)
    for tap in range(27):
        dz, dy, dx = tap // 9, tap // 3 % 3, tap % 3
        y = y + xp[dz:dz + n, dy:dy + n, dx:dx + n] @ w[tap].T
    return y


def _grad64(case, seed):
    """Loss of the smoothed network and its parameter gradient."""
    b, coef = _dense_system(case, seed)
    theta = torch.from_numpy(np.load(NET, allow_pickle=False)).cuda().double().requires_grad_(True)
    apply, diag = _operator(coef)
    mask = (coef != 0).double()
    inv = mask * (2.0 / 3.0) / diag.clamp(min=1)
    z1 = inv * b
    r1 = mask * (b - apply(z1))
    scale = torch.sqrt((r1 ** 2).sum() / mask.sum())
    at = 0
    params = []
    for cin, cout in ((16, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16)):
        w = theta[at:at + 27 * cin * cout].reshape(27, cout, cin)
        at += 27 * cin * cout
        params.append((w, theta[at:at + cout]))
        at += cout
    head, hb = theta[at:at + 16], theta[at + 16]

    def any2(m):
        n = m.shape[0] // 2
        return m.reshape(n, 2, n, 2, n, 2).amax(dim=(1, 3, 5))

    def pool(x):
        n = x.shape[0] // 2
        return x.reshape(n, 2, n, 2, n, 2, -1).mean(dim=(1, 3, 5))

    def up(x):
        return x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

    m = [mask, any2(mask), any2(any2(mask))]

    def layer(i, x, level):
        return torch.relu(_conv(x, *params[i])) * m[level][..., None]

    x0 = torch.zeros(*mask.shape, 16, dtype=torch.float64, device="cuda")
    x0[..., 0] = r1 / scale
    x0[..., 1] = mask
    b0 = layer(1, layer(0, x0, 0), 0)
    b1 = layer(3, layer(2, pool(b0), 1), 1)
    b2 = layer(5, layer(4, pool(b1), 2), 2)
    d1 = layer(7, layer(6, torch.cat([up(b2), b1], -1), 1), 1)
    d0 = layer(9, layer(8, torch.cat([up(d1), b0], -1), 0), 0)
    x = z1 + mask * scale * (d0 @ head + hb)
    z = x + inv * (b - apply(x))
    loss = ((mask * (apply(z) - b)) ** 2).sum() / (b ** 2).sum()
    loss.backward()
    return float(loss.detach()), theta.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "transfer":
        if case["n"] > 1 << 25:
            return None
        f = _Flip64(case, _cloud(case, seed))
        f.transfer()
        return [_tiled(a) for a in f.F]
    if kind in ("step", "frame", "host"):
        if not _fields(case) or kind in ("step", "frame") and case["nx"] * case["ny"] * case["nz"] > 1 << 22:
            return None
        frame = kind == "frame"
        f = _Flip64(case, _scene(case, seed, sphere=frame), _solid(case) if frame else None)
        f.transfer()
        if frame:
            f.set_box(*_paddle(0.0))
            fast = max(float(v.abs().max()) for v in f.v)
            dt = min(case["frame"], 0.5 * f.h / fast)
            f.step(dt)
            if dt < case["frame"]:
                f.move(dt)
                f.transfer()
                f.step(case["frame"] - dt)
        else:
            f.step(case.get("dt", 1.0 / 240.0))
        if kind == "host":
            # in the order of the cells that the particles came from
            c = [torch.floor(q).long() for q in f.q]
            nb = [n // 8 for n in f.size]
            key = (((c[2] >> 3) * nb[1] + (c[1] >> 3)) * nb[0] + (c[0] >> 3)) * 512 + (c[2] & 7) * 64 + (c[1] & 7) * 8 + (c[0] & 7)
            order = torch.sort(key, stable=True)[1]
            f.move(1.0 / 240.0)
            return [a[order] for a in f.x + f.v]
        return [_tiled(a) for a in f.F]
    if kind == "learned":
        c = _learned_scene(case)
        f = _Flip64(c, _scene(c, seed, sphere=True), _solid(c))
        f.transfer()
        f.system(1.0 / 240.0)
        f.solve()
        return _slots(f.p, f.fluid)
    if kind == "grad":
        return _grad64(case, seed)
    return None  # whole numbers, or FP64 already with the reference's own order of operations

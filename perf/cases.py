"""What the level-set framework is timed on: calls through its Python entry points.

Twelve listed cases and the ranges that they stand for.  Every input is made
on the GPU from a seed.  A case's "kind" says which call it is:

- "step": one dense update, SL step and curvature (levelset_step), the call of
  a solver that advances a whole window: the 2D windows of a few hundred nodes
  per axis (a pass is launch latency), the FP64 3D windows with the velocity
  as component planes or per node, the FP32 windows of the precision form.
- "batch": one step of many uneven cells packed together (Batch), as a rank
  holding many DCells takes it, after the autotuner has chosen the launches.
- "adjoint": forward and backward of a short trajectory with checkpoints
  (advect_n), the inner loop of fitting a velocity field.
- "pls": one particle level-set step: particles moved, phi advected, escaped
  particles corrected, curvature, radii adjusted.
- "band": one band-mode step without reinitialisation: the SL step at the band
  nodes, the CFL reduction, the irregular-node list, its surface quantities.
- "advect_reinit": one whole DeviceLevelSet.advect_and_reinit that passes the
  CFL threshold, so that it rebuilds phi and the band.
- "reinit": reinitialisation of a batch of level sets, with the exact fast
  marching (the default of DeviceLevelSet) or the parallel sweeps.
- "window": the velocity window taken from the fluid's array, and the output
  file's bytes of a grid.

Sizes are those of this repository's workloads (128 squared, 128, 256 and 384
cubed, cells of edge 32 to 128, 2D cells of edge 64 to 512) and odd ones
between them.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.utils.checkpoint

import dcell_amd as D
from dcell_amd import adjoint as A
from dcell_amd import formats as F
from dcell_amd import metrics as M
from dcell_amd import pls as PL
from dcell_amd.advect import DeviceLevelSet
from dcell_amd.batch import Batch

DEV = "cuda:0"
DTYPES = {"f64": torch.float64, "f32": torch.float32}
BAND, INF = 6.0, 7.5  # the reference's band width and far value, in cells


def listed():
    return [
        # the 2D slotted-disk class of problem: two small kernels, so latency
        {"name": "step2d_f64_128", "kind": "step", "nx": 128, "ny": 128, "nz": 1, "dtype": "f64", "interp": "cubic",
         "backtrace": "rk2", "planes": False, "flow": "rotation"},
        # the main double-precision workload: 256 cubed, component planes
        {"name": "step3d_f64_planes_256", "kind": "step", "nx": 256, "ny": 256, "nz": 256, "dtype": "f64",
         "interp": "cubic", "backtrace": "rk2", "planes": True, "flow": "deformation"},
        # the reference's own scheme on a window of odd extents, per-node velocity
        {"name": "step3d_f64_euler_odd", "kind": "step", "nx": 211, "ny": 173, "nz": 149, "dtype": "f64",
         "interp": "linear", "backtrace": "euler", "planes": False, "flow": "deformation"},
        # the precision form's window
        {"name": "step3d_f32_384", "kind": "step", "nx": 384, "ny": 384, "nz": 384, "dtype": "f32", "interp": "cubic",
         "backtrace": "rk2", "planes": False, "flow": "deformation"},
        # many cells at once, single precision, half of the 512-cell batch
        {"name": "batch3d_f32_256", "kind": "batch", "dim": 3, "cells": 256, "lo": 32, "hi": 128, "dtype": "f32",
         "interp": "cubic", "backtrace": "rk2"},
        # 2D cells in double precision
        {"name": "batch2d_f64_256", "kind": "batch", "dim": 2, "cells": 256, "lo": 64, "hi": 512, "dtype": "f64",
         "interp": "cubic", "backtrace": "rk2"},
        # velocity fitting: ten steps forward and back, a checkpoint every five
        {"name": "adjoint_f32_128", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 128, "dtype": "f32",
         "interp": "cubic", "backtrace": "rk2", "steps": 10, "every": 5},
        # a particle level-set step
        {"name": "pls_f32_256", "kind": "pls", "nx": 256, "ny": 256, "nz": 256, "dtype": "f32", "per_cell": 32},
        # band mode between reinitialisations
        {"name": "band_f64_256", "kind": "band", "nx": 256, "ny": 256, "nz": 256, "interp": "linear",
         "backtrace": "euler"},
        # band mode, a step that reinitialises
        {"name": "advect_reinit_256", "kind": "advect_reinit", "nx": 256, "ny": 256, "nz": 256, "reinit": "parallel"},
        # a rank's cells rebuilt in the reference's own order
        {"name": "reinit_exact_24", "kind": "reinit", "cells": 24, "lo": 32, "hi": 64, "method": "exact"},
        # the steps either side: velocity in, grid file out
        {"name": "window_f64_256", "kind": "window", "nx": 256, "ny": 256, "nz": 256, "dtype": "f64", "planes": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _axes(rng, lo, hi):
    """Three extents around one log-uniform size, odd ones among them."""
    n = _log(rng, lo, hi)
    return {k: max(lo, min(hi, int(n * rng.uniform(0.75, 1.25)))) for k in ("nx", "ny", "nz")}


def _extents(case):
    return [case["nx"], case["ny"], case["nz"]]


def draw(rng: random.Random):
    kind = rng.choice(["step2d", "step3d", "step3d", "batch", "batch", "adjoint", "pls", "band", "advect_reinit",
                       "reinit", "window"])
    dtype = rng.choice(["f64", "f32"])
    interp, backtrace = rng.choice([("cubic", "rk2"), ("cubic", "rk2"), ("cubic", "euler"), ("linear", "rk2"),
                                    ("linear", "euler")])
    flow = rng.choice(["deformation", "fourier"])
    if kind == "step2d":
        n = _axes(rng, 32, 1024)
        return {"kind": "step", **n, "nz": 1, "dtype": dtype, "interp": interp, "backtrace": backtrace,
                "planes": rng.random() < 0.3, "flow": rng.choice(["rotation", "fourier"])}
    if kind == "step3d":
        return {"kind": "step", **_axes(rng, 32, 256), "dtype": dtype, "interp": interp, "backtrace": backtrace,
                "planes": rng.random() < 0.5, "flow": flow}
    if kind == "batch":
        if rng.random() < 0.5:
            return {"kind": "batch", "dim": 3, "cells": _log(rng, 4, 96), "lo": 32, "hi": 128, "dtype": dtype,
                    "interp": interp, "backtrace": backtrace}
        return {"kind": "batch", "dim": 2, "cells": _log(rng, 4, 256), "lo": 64, "hi": 512, "dtype": dtype,
                "interp": interp, "backtrace": backtrace}
    if kind == "adjoint":
        return {"kind": "adjoint", **_axes(rng, 32, 128), "dtype": dtype, "interp": interp,
                "backtrace": backtrace, "steps": rng.randint(2, 10), "every": rng.randint(1, 5)}
    if kind == "pls":
        return {"kind": "pls", **_axes(rng, 48, 224), "dtype": dtype, "per_cell": rng.choice([16, 24, 32])}
    if kind == "band":
        return {"kind": "band", **_axes(rng, 48, 256), "interp": interp, "backtrace": backtrace}
    if kind == "advect_reinit":
        method = rng.choice(["parallel", "parallel", "exact"])
        return {"kind": "advect_reinit", **_axes(rng, 48, 64 if method == "exact" else 256), "reinit": method}
    if kind == "reinit":
        method = rng.choice(["parallel", "exact"])
        return {"kind": "reinit", "cells": _log(rng, 2, 24 if method == "exact" else 64), "lo": 32,
                "hi": 56 if method == "exact" else 96, "method": method}
    return {"kind": "window", **_axes(rng, 32, 256), "dtype": dtype, "planes": rng.random() < 0.5}


# ------------------------------------------------------------------- inputs
def _coords(n, h, shift=None):
    """Broadcastable node coordinates (x, y[, z]) of a window, shifted by cells."""
    dim = 2 if n[2] < 2 else 3
    out = []
    for a in range(dim):
        c = torch.arange(n[a], device=DEV, dtype=torch.float64) * h
        if shift is not None and shift == a:
            c = c - 0.5 * h
        out.append(c.view([-1 if d == dim - 1 - a else 1 for d in range(dim)]))
    return out


def _shape(n):
    return (n[1], n[0]) if n[2] < 2 else (n[2], n[1], n[0])


def _window(n, p=(0, 0, 0)):
    h = 1.0 / (max(n) - 1)
    return D.GridWindow(tuple(p), tuple(n), (h, h, h)), h


def _sphere(n, h, g):
    """Signed distance in cells to a sphere (circle) that lies well inside the window."""
    dim = 2 if n[2] < 2 else 3
    ext = [(n[a] - 1) * h for a in range(dim)]
    small = min(ext)
    center = [ext[a] * 0.5 + small * g.uniform(-0.08, 0.08) for a in range(dim)]
    r = small * g.uniform(0.2, 0.28)
    d2 = sum((c - center[a]) ** 2 for a, c in enumerate(_coords(n, h)))
    return ((torch.sqrt(d2) - r) / h).contiguous()


def _flow(n, h, flow, g):
    """MAC velocity, shaped (window, dim) in float64, and its time step."""
    dim = 2 if n[2] < 2 else 3
    vel = torch.zeros(_shape(n) + (dim,), dtype=torch.float64, device=DEV)
    if flow == "rotation":
        x, y = _coords(n, h, 0)
        vel[..., 0] = 2 * math.pi * (0.5 - y)
        x, y = _coords(n, h, 1)
        vel[..., 1] = 2 * math.pi * (x - 0.5)
        return vel, h / (2 * math.pi)
    if flow == "deformation":
        # LeVeque's field at a time of its period, with dt = h
        amp = math.cos(math.pi * g.uniform(0.0, 0.3))
        s2 = [[torch.sin(2 * math.pi * c) for c in _coords(n, h, a)] for a in range(3)]
        sq = [torch.sin(math.pi * _coords(n, h, a)[a]) ** 2 for a in range(3)]
        vel[..., 0] = 2 * amp * sq[0] * s2[0][1] * s2[0][2]
        vel[..., 1] = -amp * s2[1][0] * sq[1] * s2[1][2]
        vel[..., 2] = -amp * s2[2][0] * s2[2][1] * sq[2]
        return vel, h
    for _ in range(6):  # six divergence-free Fourier modes
        while True:
            k = g.integers(-3, 4, size=dim)
            if np.abs(k).max() >= 1:
                break
        a = g.normal(0.0, 0.5, size=dim)
        a = a - k * (a @ k) / (k @ k)
        theta = g.uniform(0, 2 * math.pi)
        for c in range(dim):
            xs = _coords(n, h, c)
            vel[..., c] += float(a[c]) * torch.sin(2 * math.pi * sum(float(k[d]) * xs[d] for d in range(dim)) + theta)
    return vel, 0.7 * h / max(float(vel.abs().max()), 1e-12)


def _planes(vel):
    return vel.movedim(-1, 0).contiguous()


def _particles(phi, win, per_cell, dtype, seed):
    """per_cell particles around every node with |phi| < 3, signed radii from
    phi there, then moved a little, as earlier steps would have left them."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    nodes = (phi.abs() < 3).nonzero()
    pos = nodes.flip(1).double().repeat_interleave(per_cell, 0)
    pos = pos + torch.rand(pos.shape, generator=g, device=DEV, dtype=torch.float64) - 0.5
    hi = torch.tensor(win.n, device=DEV, dtype=torch.float64) - 1.000001
    pos = torch.minimum(pos.clamp_min(0.0), hi)
    base, w = _linear_weights(pos, win.n)
    ph = _gather(phi.double().reshape(-1), win.n, base, w)
    r = torch.where(ph >= 0, 1.0, -1.0) * ph.abs().clamp(0.1, 0.5)
    pos = pos + 0.1 * torch.randn(pos.shape, generator=g, device=DEV, dtype=torch.float64)
    pos = torch.minimum(pos.clamp_min(0.0), hi)
    return torch.cat([pos, r[:, None]], 1).to(dtype).contiguous()


def _edges(case):
    """The cells' edges, log-uniform; they belong to the case, not to the seed."""
    g = np.random.Generator(np.random.Philox(4))
    return np.rint(np.exp(g.uniform(math.log(case["lo"]), math.log(case["hi"]), size=case["cells"]))).astype(int)


def _batch_cells(case, g):
    """Windows, FP64 fields and time steps of a batch's cells: perturbed
    spheres (circles) in Fourier flows at CFL 0.7."""
    for e in _edges(case):
        n = [int(e), int(e), int(e) if case["dim"] == 3 else 1]
        win, h = _window(n)
        vel, dt = _flow(n, h, "fourier", g)
        yield win, _sphere(n, h, g), vel, dt


def _level_sets(case, g):
    """(phi, win, records, count) of a reinitialisation batch: spheres whose
    phi is 1.5 times the distance, with their irregular-node records."""
    edges = [int(e) for e in _edges(case)]
    flat = torch.empty(sum(e ** 3 for e in edges), dtype=torch.float64, device=DEV)
    cells, at = [], 0
    for e in edges:
        win, h = _window([e] * 3)
        phi = flat[at:at + e ** 3].view(win.shape)
        at += e ** 3
        phi.copy_(1.5 * _sphere([e] * 3, h, g))
        cells.append((phi, win) + _records(phi, win)[1:])
    return flat, cells


def _records(phi, win):
    band, _ = M.band_compact(phi, win, BAND)
    band = band.contiguous()
    rec = torch.empty(max(10 * band.shape[0], 1) * M.IRREGULAR_DTYPE.itemsize, dtype=torch.uint8, device=DEV)
    count = M.irregular_nodes_into(phi, win, band, rec)
    return band, rec, count


def prepare(case, seed):
    g = np.random.Generator(np.random.Philox(seed))
    kind = case["kind"]
    s = {"case": case}
    if kind == "batch":
        dtype = DTYPES[case["dtype"]]
        cells = list(_batch_cells(case, g))
        b = Batch([c[0] for c in cells], dtype=dtype, interp=case["interp"], backtrace=case["backtrace"])
        s.update(batch=b, phi0=b.new_field(), phi=b.new_field(), kappa=b.new_field(), vel=b.new_field(case["dim"]))
        for i, (_, phi, vel, _) in enumerate(cells):
            b.cell(s["phi0"], i).copy_(phi)
            b.cell(s["vel"], i, case["dim"]).copy_(vel)
        b.set_dt([c[3] for c in cells])
        b.autotune(s["phi0"], s["phi"], s["kappa"], s["vel"], reps=2)
        return s
    if kind == "reinit":
        s["phi"], s["cells"] = _level_sets(case, g)
        s["bands"] = torch.zeros((s["phi"].numel() // 2, 3), dtype=torch.int32, device=DEV)
        return s
    n = _extents(case)
    p = tuple(int(v) for v in g.integers(-5, 6, size=3)) if kind == "step" else (0, 0, 0)
    win, h = _window(n, p if n[2] >= 2 else (p[0], p[1], 0))
    s["win"] = win
    if kind == "window":
        # a window inside a fluid domain that is a little larger
        dtype = DTYPES[case["dtype"]]
        off = [int(v) for v in g.integers(0, 4, size=3)]
        big = [n[a] + 4 for a in range(3)]
        tg = torch.Generator(device=DEV).manual_seed(seed)
        s["win"] = D.GridWindow(tuple(off), tuple(n), (h, h, h))
        s["fluid"] = torch.randn((big[2], big[1], big[0], 4), generator=tg, device=DEV, dtype=dtype)
        s["grid"] = _sphere(n, h, g).to(dtype)
        s["vel"] = torch.zeros(((3,) + _shape(n)) if case["planes"] else (_shape(n) + (3,)), dtype=dtype, device=DEV)
        s["bytes"] = torch.empty(8 + 8 * win.nodes, dtype=torch.uint8, device=DEV)
        return s
    # band lists and particles are made from phi: there the case gives it and the seed the flow
    fixed = kind in ("band", "advect_reinit", "pls")
    phi = _sphere(n, h, np.random.Generator(np.random.Philox(4)) if fixed else g)
    vel, s["dt"] = _flow(n, h, case.get("flow", "fourier" if kind == "adjoint" else "deformation"), g)
    if kind in ("band", "advect_reinit"):
        s["phi0"], s["vel"] = phi, vel
        s["band"], rec, count = _records(phi, win)
        if kind == "band":
            cap = s["band"].shape[0]
            s.update(phi=torch.empty_like(phi), records=rec[:count * 88].clone(),
                     out_records=torch.zeros(cap * 88, dtype=torch.uint8, device=DEV),
                     surf=torch.zeros(cap * 104, dtype=torch.uint8, device=DEV))
        else:
            s["ls"] = DeviceLevelSet(phi.clone(), win, band_width=BAND, phi_inf=INF, reinit=case["reinit"])
            s["ls"].update_irregular_nodes()
            s["count"] = s["ls"].count
            s["buffer"] = s["ls"].records
            s["records"] = s["buffer"][:s["count"] * 88].clone()
            s["bands"] = torch.zeros((win.nodes // 2, 3), dtype=torch.int32, device=DEV)
        return s
    dtype = DTYPES[case["dtype"]]
    s["phi0"] = phi.to(dtype)
    s["vel"] = (_planes(vel) if case.get("planes") else vel).to(dtype)
    if kind == "step":
        s.update(phi=torch.empty_like(s["phi0"]), kappa=torch.empty_like(s["phi0"]))
    elif kind == "adjoint":
        s["phi0"].requires_grad_(True)
        s["vel"].requires_grad_(True)
        # the gradient of a loss that lives at the interface
        s["grad"] = (torch.clamp(1 - s["phi0"].detach().abs() / 6.0, min=0.0) * torch.sign(s["phi0"].detach())
                     ).contiguous()
    else:
        P = _particles(s["phi0"], win, case["per_cell"], dtype, seed)
        s.update(P0=P, P=torch.empty_like(P), phi=torch.empty_like(s["phi0"]), kappa=torch.empty_like(s["phi0"]),
                 ws=PL.CorrectionWorkspace(win.nodes, 8 * len(P), dtype))
    return s


# --------------------------------------------------------------------- passes
def _split_records(rec):
    """The integer and the floating fields of a buffer of records."""
    r = rec.view(-1, 88)
    return r[:, :32].view(torch.int32), r[:, 32:].view(torch.float64)


def _put(bands, *parts):
    """Band lists one after another in a buffer (their length depends on phi)."""
    at = 0
    for b in parts:
        bands[at:at + b.shape[0]].copy_(b)
        at += b.shape[0]
    return bands, at


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        return D.levelset_step(s["phi0"], s["vel"], s["win"], s["dt"], case["interp"], case["backtrace"],
                               out_phi=s["phi"], out_kappa=s["kappa"], planes=case["planes"])
    if kind == "batch":
        s["batch"].step(s["phi0"], s["phi"], s["kappa"], s["vel"])
        return s["phi"], s["kappa"]
    if kind == "adjoint":
        phi = A.advect_n(s["phi0"], s["vel"], s["win"], s["dt"], case["steps"], case["interp"], case["backtrace"],
                         checkpoint_every=case["every"])
        lam, gvel = torch.autograd.grad(phi, (s["phi0"], s["vel"]), s["grad"])
        return phi.detach(), lam, gvel
    if kind == "pls":
        win, dt = s["win"], s["dt"]
        s["P"].copy_(s["P0"])
        PL.advect_particles(s["P"], s["vel"], win, win.d, dt)
        D.advect_sl(s["phi0"], s["vel"], win, dt, "cubic", "rk2", out=s["phi"])
        PL.correct(s["P"], s["phi"], win, s["ws"])
        D.curvature(s["phi"], win, out=s["kappa"])
        PL.adjust_radii(s["P"], s["phi"], win)
        return s["P"][:, :3], s["P"][:, 3], s["phi"], s["kappa"]
    if kind == "band":
        win = s["win"]
        s["phi"].copy_(s["phi0"])
        D.advect_sl(s["phi0"], s["vel"], win, s["dt"], case["interp"], case["backtrace"], band=s["band"],
                    out=s["phi"])
        vmax = M.max_velocity(s["vel"], win, s["records"], stride_bytes=88)
        count = M.irregular_nodes_into(s["phi"], win, s["band"], s["out_records"])
        M.surface_quantities_into(s["phi"], win, s["out_records"], count, s["surf"])
        return (s["phi"], vmax, count) + _split_records(s["out_records"]) + (s["surf"].view(torch.float64),)
    if kind == "advect_reinit":
        # the state a time loop has just past the CFL threshold
        ls = s["ls"]
        ls.phi.copy_(s["phi0"])
        ls.band, ls.records, ls.count = s["band"], s["buffer"], s["count"]
        ls.records[:s["records"].numel()].copy_(s["records"])
        ls.cfl_count, ls.advect_count = ls.cfl_thres, 0
        ls.advect_and_reinit(s["vel"], s["dt"])
        return (ls.phi, ls.max_vel) + _put(s["bands"], ls.band)
    if kind == "reinit":
        # phi enters through its signs only, so a pass can be repeated
        if case["method"] == "exact":
            bands = M.reinitialize(s["cells"], BAND, INF)
        else:
            bands, _ = M.reinitialize_parallel(s["cells"], BAND, INF)
        return (s["phi"],) + _put(s["bands"], *bands)
    vel = D.get_velocity(s["fluid"], s["win"], out=s["vel"], planes=case["planes"])
    return vel, F.real64_pack(s["grid"], out=s["bytes"])


# ----------------------------------------------------------------------- work
def _size(dtype):
    return 8 if dtype == "f64" else 4


def _sl_flops(dim, interp, backtrace):
    """Multiplies and adds of one node's SL update."""
    cells = 4 if interp == "cubic" else 2
    gather = sum(2 * cells ** d for d in range(1, dim + 1)) + (dim * 12 if interp == "cubic" else 0)
    mac = dim * 3 * (2 ** dim - 1)
    return 4 * dim + gather + (mac + 4 * dim if backtrace == "rk2" else 0)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        nodes, dim, b = float((_edges(case) ** case["dim"]).sum()), case["dim"], _size(case["dtype"])
        return {"bytes": nodes * b * (3 + dim), "flops": nodes * (_sl_flops(dim, case["interp"], case["backtrace"])
                                                                 + (60 if dim == 3 else 25))}
    if kind == "reinit":
        n = _edges(case).astype(float)
        band = float((4 * math.pi * (0.24 * n) ** 2 * 8).sum())
        return {"bytes": float((n ** 3).sum()) * 16 + band * (12 + 30), "flops": band * 120}
    n = _extents(case)
    nodes = float(n[0] * n[1] * n[2])
    dim = 2 if n[2] < 2 else 3
    if kind == "window":
        b = _size(case["dtype"])
        return {"bytes": nodes * (4 * b + 3 * b + b + 8), "flops": nodes}
    band = 4 * math.pi * (0.24 * min(n)) ** 2 * 12
    if kind == "band":
        return {"bytes": nodes * 16 + band * 12 * 2 + band * (8 + 24) + band * 0.5 * (88 * 3 + 104),
                "flops": band * 300}
    if kind == "advect_reinit":
        return {"bytes": nodes * (16 + 16) + band * (12 * 3 + 32) + band * 0.5 * 88 * 3, "flops": band * 400}
    b = _size(case["dtype"])
    if kind == "step":
        sl = _sl_flops(dim, case["interp"], case["backtrace"])
        return {"bytes": nodes * b * (3 + dim), "flops": nodes * (sl + (60 if dim == 3 else 25))}
    sl = _sl_flops(3, case.get("interp", "cubic"), case.get("backtrace", "rk2"))
    if kind == "adjoint":
        # phi at both ends, the incoming gradient, the velocity, both gradients
        return {"bytes": nodes * b * (4 + 3 + 3), "flops": nodes * case["steps"] * 4 * sl}
    parts = 4 * math.pi * (0.24 * min(n)) ** 2 * 6 * case["per_cell"]
    return {"bytes": nodes * b * 6 + parts * 8 * b, "flops": nodes * (sl + 60) + parts * 200}


# ------------------------------------------------- the same in 64 bits (torch)
def _split(x, lo, hi, top):
    """Clamp to [lo, hi], base index at most top, fraction."""
    x = x.clamp(lo, hi)
    b = torch.floor(x).clamp_max(top)
    return b.long(), x - b


def _linear_weights(pos, n):
    base, w = [], []
    for a in range(pos.shape[1]):
        b, f = _split(pos[:, a], 0.0, float(n[a] - 1), n[a] - 2)
        base.append(b)
        w.append([1 - f, f])
    return base, w


def _cubic_weights(pos, n):
    base, w = [], []
    for a in range(pos.shape[1]):
        b, t = _split(pos[:, a], 1.0, float(n[a] - 2), n[a] - 3)
        base.append(b - 1)
        w.append([0.5 * (2 * t ** 2 - t ** 3 - t), 0.5 * (3 * t ** 3 - 5 * t ** 2 + 2),
                  0.5 * (4 * t ** 2 + t - 3 * t ** 3), 0.5 * (t ** 3 - t ** 2)])
    return base, w


def _gather(flat, n, base, w):
    """Sum of a separable stencil over a flat field of extents n (x fastest)."""
    dim = len(base)
    stride = [1, n[0], n[0] * n[1]][:dim]
    corner = sum(base[a] * stride[a] for a in range(dim))

    def level(a, off):
        if a < 0:
            return flat.index_select(0, corner + off)
        return sum(w[a][i] * level(a - 1, off + i * stride[a]) for i in range(len(w[a])))

    return level(dim - 1, 0)


def _mac(vel, pos, n):
    """MAC velocity at local positions; vel: one flat field per component."""
    dim = pos.shape[1]
    plain, shifted = [], []
    for a in range(dim):
        x = pos[:, a].clamp(0.0, float(n[a] - 2))
        b0, b1 = torch.floor(x), torch.floor(x + 0.5)
        plain.append((b0.long(), x - b0))
        shifted.append((b1.long(), x - b1 + 0.5))
    out = []
    for c in range(dim):
        pick = [shifted[a] if a == c else plain[a] for a in range(dim)]
        out.append(_gather(vel[c], n, [q[0] for q in pick], [[1 - q[1], q[1]] for q in pick]))
    return torch.stack(out, 1)


def _components(vel, planes, dim):
    return [vel[c].double().reshape(-1) if planes else vel[..., c].double().reshape(-1) for c in range(dim)]


def _sl_nodes(phi, vel, pos, n, c, interp, backtrace):
    v = _mac(vel, pos, n)
    if backtrace == "rk2":
        v = _mac(vel, pos - 0.5 * c * v, n)
    base, w = (_cubic_weights if interp == "cubic" else _linear_weights)(pos - c * v, n)
    return _gather(phi, n, base, w)


def _interior(n, lo, hi):
    """Flat indices and local positions of interior nodes of slabs [lo, hi) of the slowest axis."""
    dim = 2 if n[2] < 2 else 3
    last = dim - 1
    ax = [torch.arange(2, n[a] - 2, device=DEV) for a in range(dim)]
    ax[last] = torch.arange(max(2, lo), min(n[last] - 2, hi), device=DEV)
    grid = torch.meshgrid(*reversed(ax), indexing="ij")
    pos = torch.stack([q.reshape(-1) for q in reversed(grid)], 1)
    stride = [1, n[0], n[0] * n[1]]
    return sum(pos[:, a] * stride[a] for a in range(dim)), pos.double()


def _sl(phi, vel, n, c, interp, backtrace):
    """One dense SL step of a flat FP64 field; the two outer layers carry over."""
    dim = 2 if n[2] < 2 else 3
    out = phi.clone()
    per = max(1, 4_000_000 // (n[0] * (n[1] if dim == 3 else 1)))
    for lo in range(0, n[dim - 1], per):
        idx, pos = _interior(n, lo, lo + per)
        if idx.numel():
            out = out.index_put((idx,), _sl_nodes(phi, vel, pos, n, c, interp, backtrace))
    return out


def _curvature(phi, win):
    """The 19-point (9-point in 2D) curvature of a window, 0 on its outer layer."""
    dim = win.dim
    p = phi.double().view(win.shape)
    out = torch.zeros_like(p)

    def at(off):
        return p[tuple(slice(1 + off[dim - 1 - d], p.shape[d] - 1 + off[dim - 1 - d]) for d in range(dim))]

    def e(a, s=1):
        return [s if q == a else 0 for q in range(dim)]

    def add(x, y):
        return [i + j for i, j in zip(x, y)]

    h = win.d
    first = [(at(e(a)) - at(e(a, -1))) / (2 * h[a]) for a in range(dim)]
    second = [(at(e(a)) - 2 * at([0] * dim) + at(e(a, -1))) / h[a] ** 2 for a in range(dim)]
    g2 = sum(f * f for f in first)
    c = sum(first[a] ** 2 * sum(second[b] for b in range(dim) if b != a) for a in range(dim))
    for a in range(dim):
        for b in range(a + 1, dim):
            cross = (at(add(e(a), e(b))) + at(add(e(a, -1), e(b, -1))) - at(add(e(a), e(b, -1)))
                     - at(add(e(a, -1), e(b)))) / (4 * h[a] * h[b])
            c = c - 2 * first[a] * first[b] * cross
    k = c / torch.sqrt(g2 * g2 * g2)
    out[(slice(1, -1),) * dim] = torch.where(torch.isnan(k), 0.0, k)
    return out


def _exact_step(phi0, vel, win, dt, interp, backtrace, planes):
    comps = _components(vel, planes, win.dim)
    return _sl(phi0.double().reshape(-1), comps, win.n, dt / win.d[0], interp, backtrace).view(win.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "reinit":
        return None  # the order of acceptance is the algorithm; no formula gives it
    if kind == "batch":
        g = np.random.Generator(np.random.Philox(seed))
        dtype = DTYPES[case["dtype"]]
        phis, kappas = [], []
        for win, phi, vel, dt in _batch_cells(case, g):
            q = _exact_step(phi.to(dtype), vel.to(dtype), win, dt, case["interp"], case["backtrace"], False)
            phis.append(q.reshape(-1))
            kappas.append(_curvature(q, win).reshape(-1))
        return torch.cat(phis), torch.cat(kappas)
    s = prepare(case, seed)
    win = s["win"]
    if kind == "window":
        off, n = win.p, win.n
        v = s["fluid"][off[2]:off[2] + n[2], off[1]:off[1] + n[1], off[0]:off[0] + n[0], 1:].double()
        return (_planes(v) if case["planes"] else v.contiguous()), None
    if kind == "step":
        phi = _exact_step(s["phi0"], s["vel"], win, s["dt"], case["interp"], case["backtrace"], case["planes"])
        return phi, _curvature(phi, win)
    if kind == "adjoint":
        phi0 = s["phi0"].detach().double().requires_grad_(True)
        vel = s["vel"].detach().double().requires_grad_(True)

        def one(phi, vel):
            return _sl(phi, [vel[..., c].reshape(-1) for c in range(3)], win.n, s["dt"] / win.d[0], case["interp"],
                       case["backtrace"])

        phi = phi0.reshape(-1)
        for _ in range(case["steps"]):
            phi = torch.utils.checkpoint.checkpoint(one, phi, vel, use_reentrant=False)
        phi = phi.view(win.shape)
        lam, gvel = torch.autograd.grad(phi, (phi0, vel), s["grad"].double())
        return phi.detach(), lam, gvel
    if kind == "pls":
        comps = _components(s["vel"], False, 3)
        x = s["P0"][:, :3].double()
        c = s["dt"] / win.d[0]
        v = _mac(comps, x + 0.5 * c * _mac(comps, x, win.n), win.n)
        return x + c * v, None, None, None
    # band mode: phi at the band nodes, the rest carried over; the list has no formula of its own
    if kind == "band":
        comps = _components(s["vel"], False, 3)
        idx = s["band"].long()
        flat = (idx[:, 2] * win.n[1] + idx[:, 1]) * win.n[0] + idx[:, 0]
        phi = s["phi0"].reshape(-1).clone()
        phi[flat] = _sl_nodes(s["phi0"].reshape(-1), comps, idx.double(), win.n, s["dt"] / win.d[0], case["interp"],
                              case["backtrace"])
        return phi.view(win.shape), None, None, None, None, None
    return None

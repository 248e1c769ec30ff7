"""Performance cases of the PBF step: what a user of this package has it do.

A pass is one call of a public entry point on a particle state, from the smallest
scenes (latency, launches) to the 16.7M-particle dam break:

  noalloc  pbd_compute_noalloc on the caller's device arrays, stream-ordered on
           the caller's stream: many small steps inside another GPU program
  frame    Context.step(1, graph=True) and sync, the simulation loop: a dam
           break's first moments ("column": the block still at rest density) or
           its spread-out, splashing flow ("splash": a pool, waves and spray,
           most 2 x 4 x 4-cell blocks nearly empty), with or without granular
           solids and friction
  refcfg   the same loop under the parameters of configs/reference.txt: the
           reference's own formulas, wide kernels and two-cell stencil
  batch    Batch.step and the read-back of every scene's positions, as a data
           generation or control loop over many uneven scenes does
  adjoint  one iteration of an optimisation through the simulator: upload the
           initial state, pbd_adj_forward, the loss adjoint from the final
           positions, pbd_adj_backward

Every frame / refcfg / noalloc pass starts from the same state (a program that
resets its scene): the state is copied into the context's device buffers, in the
particle order that a previous step leaves (sorted by cell).  All inputs come
from the seed alone.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "pbd-simulation-framework-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import pbdfluid as F  # noqa: E402
from pbdfluid.workloads import uneven_dam_breaks  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ---------------------------------------------------------------------------
# Cases.  w x h x d: the dam break's lattice; the box is length x w, h, d lattice
# spacings; n particles of it are there (ragged counts leave vacancies).
def listed():
    return [
        # the smallest scenes, stepped inside another program: launches and latency
        {"name": "noalloc_2k", "kind": "noalloc", "n": 2197, "w": 13, "h": 13, "d": 13, "length": 2, "flow": "column"},
        # the largest scene of that entry point, odd count, spread-out
        {"name": "noalloc_30k", "kind": "noalloc", "n": 30011, "w": 32, "h": 32, "d": 32, "length": 2,
         "flow": "splash"},
        # the reference's own CPU-sized dam break (configs/dam_break_32k.txt)
        {"name": "frame_32k", "kind": "frame", "n": 32768, "w": 32, "h": 32, "d": 32, "length": 2, "flow": "column",
         "solids": 0.0},
        # a mid-sized scene late in its run, ragged in count and box
        {"name": "splash_211k", "kind": "frame", "n": 211003, "w": 61, "h": 59, "d": 60, "length": 3, "flow": "splash",
         "solids": 0.0},
        # the headline dam break (configs/dam_break_1m.txt), early and late
        {"name": "column_1m", "kind": "frame", "n": 1048576, "w": 64, "h": 128, "d": 128, "length": 4,
         "flow": "column", "solids": 0.0},
        {"name": "splash_1m", "kind": "frame", "n": 1048576, "w": 64, "h": 128, "d": 128, "length": 4,
         "flow": "splash", "solids": 0.0},
        # granular solids with friction among the fluid (configs/mixed_16m.txt at a common size)
        {"name": "mixed_500k", "kind": "frame", "n": 500009, "w": 80, "h": 80, "d": 80, "length": 2, "flow": "column",
         "solids": 0.3},
        # the largest shipped scene (configs/dam_break_16m.txt)
        {"name": "column_16m", "kind": "frame", "n": 16777216, "w": 256, "h": 256, "d": 256, "length": 2,
         "flow": "column", "solids": 0.0},
        # the reference's shipped parameters and spawn box (configs/reference.txt)
        {"name": "reference_14k", "kind": "refcfg", "n": 13824, "side": 24},
        # many uneven scenes at once
        {"name": "batch_64", "kind": "batch", "scenes": 64, "lo": 2048, "hi": 32768, "frames": 4},
        # gradients: the adjoint scene (configs/adjoint_64k.txt) and one with solids and friction
        {"name": "adjoint_64k", "kind": "adjoint", "n": 65536, "w": 64, "h": 32, "d": 32, "length": 2,
         "flow": "column", "solids": 0.0, "frames": 1},
        {"name": "adjoint_mixed_250k", "kind": "adjoint", "n": 250007, "w": 63, "h": 63, "d": 63, "length": 2,
         "flow": "column", "solids": 0.3, "frames": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["noalloc", "frame", "frame", "frame", "mixed", "refcfg", "batch", "adjoint"])
    if kind == "refcfg":
        side = rng.randint(8, 36)
        return {"kind": kind, "n": side ** 3 - rng.randint(0, side), "side": side}
    if kind == "batch":
        return {"kind": kind, "scenes": _log_int(rng, 8, 160), "lo": 2048, "hi": _log_int(rng, 4096, 32768),
                "frames": rng.randint(2, 6)}
    lo, hi = {"noalloc": (256, 30000), "frame": (3000, 4000000), "mixed": (20000, 1000000),
              "adjoint": (4000, 250000)}[kind]
    n = _log_int(rng, lo, hi)
    side = n ** (1.0 / 3.0)
    w = max(4, int(round(side * math.exp(rng.uniform(-0.4, 0.3)))))
    h = max(4, int(round(side * math.exp(rng.uniform(-0.2, 0.2)))))
    d = int(math.ceil(n / (w * h)))
    if kind == "noalloc":  # its cell table holds a grid of 32 x 32 x 32 cells
        w = h = min(31, max(w, int(math.ceil(math.sqrt(n / 60.0)))))
        d = int(math.ceil(n / (w * h)))
        case = {"kind": kind, "length": 2, "flow": rng.choice(["column", "splash"])}
    elif kind == "adjoint":
        case = {"kind": kind, "length": 2, "flow": "column", "solids": rng.choice([0.0, 0.0, 0.3]), "frames": 1}
    elif kind == "mixed":
        case = {"kind": "frame", "length": rng.randint(2, 3), "flow": "column",
                "solids": round(rng.uniform(0.1, 0.5), 2)}
    else:
        case = {"kind": kind, "length": rng.randint(2, 4), "flow": rng.choice(["column", "splash"]), "solids": 0.0}
    return {**case, "n": n, "w": w, "h": h, "d": d}


# ---------------------------------------------------------------------------
# Scenes.  The dam-break configs' solver (h = cell = 0.1, spacing 0.05, dt = 1/120
# per substep, 4 iterations), one substep per frame except in the adjoint cases.
S, CELL = 0.05, 0.1
DAM = dict(variant=1, kw=1, cell=CELL, origin=0.0, diameter=0.05, hp=0.1, hs=0.1, dq=0.02, k_scorr=0.1, n_scorr=4,
           stiffness=0.3, eps=600.0, gravity=-9.81, iters=4, c_visc=0.01, e_vort=0.0005, cap=512, mu_s=0.0, mu_k=0.0)
REF = dict(variant=0, kw=2, cell=1.0, origin=0.0, diameter=1.0, hp=4.1, hs=6.1, dq=1.22, k_scorr=0.2, n_scorr=4,
           stiffness=0.3, eps=1e-4, gravity=-29.82, iters=1, c_visc=0.0001, e_vort=1.0, cap=512, mu_s=0.0, mu_k=0.0,
           rho0=1200.0, dt=0.01, bmin=[1.5] * 3, bmax=[62.5] * 3, dims=[128] * 3)


def _constants(case):
    """The step's parameters as plain numbers."""
    if case["kind"] == "refcfg":
        return dict(REF)
    c = dict(DAM)
    box = [case["length"] * case["w"] * S, case["h"] * S, case["d"] * S]
    c["bmin"], c["bmax"] = [0.0] * 3, [float(np.float32(b)) for b in box]
    c["dims"] = [int(math.ceil(b / CELL - 1e-6)) for b in box]
    c["dt"] = float(np.float32(1.0 / 60.0) / np.float32(2.0))
    if case.get("solids"):
        c["mu_s"], c["mu_k"] = 0.5, 0.4
    m = int(math.ceil(c["hp"] / S)) + 1  # rest density of the lattice
    k = np.arange(-m, m + 1) * S
    r2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, :] ** 2
    c["rho0"] = float(315.0 / (64.0 * math.pi * c["hp"] ** 9) * (np.maximum(c["hp"] ** 2 - r2, 0.0) ** 3).sum())
    return c


def _params(case):
    """The same as a parameter set of the package."""
    c = _constants(case)
    p = F.load_params(F.config_path("reference" if case["kind"] == "refcfg" else "dam_break_32k"))
    p.box_spawn_in_the_beginning = 0
    if case["kind"] == "refcfg":
        return p
    p.rest_density, p.rest_density_from_lattice = c["rho0"], 0
    if case["kind"] != "adjoint":
        p.delta_t, p.substeps = p.delta_t / p.substeps, 1
    for a in range(3):
        p.bounds_max[a], p.grid_dims[a] = c["bmax"][a], c["dims"][a]
    p.friction_static, p.friction_kinetic = c["mu_s"], c["mu_k"]
    return p


def _cells(c, pos):
    """Cell coordinates of float32 positions, in float32 as the step takes them."""
    inv = float(np.float32(1.0) / np.float32(c["cell"]))
    ijk = torch.floor((pos[:, :3] - c["origin"]) * inv)
    hi = torch.tensor(c["dims"], device=pos.device, dtype=ijk.dtype) - 1
    return torch.minimum(torch.clamp(ijk, min=0.0), hi).long()


def _morton(ijk):
    key = torch.zeros(ijk.shape[0], dtype=torch.long, device=ijk.device)
    for b in range(10):
        for a in range(3):  # x at bit 3b + 2, y at 3b + 1, z at 3b
            key |= ((ijk[:, a] >> b) & 1) << (3 * b + 2 - a)
    return key


def _predict32(c, x, v, f):
    """The predicted positions in float32: forces, then the clamp to the enclosure."""
    dt = float(np.float32(c["dt"]))
    g = torch.zeros(3, device=x.device)
    g[1] = float(np.float32(c["gravity"]) * np.float32(c["dt"]))
    v = v + g
    p = x + (v + f * dt) * dt
    lo = torch.tensor(c["bmin"], device=x.device, dtype=torch.float32)
    hi = torch.tensor(c["bmax"], device=x.device, dtype=torch.float32)
    inset = float(np.float32(0.001))
    return torch.where(p < lo, lo + inset, torch.where(p > hi, hi - inset, p))


def _state(case, seed):
    """Positions, velocities, forces (n x 4 float32 on the GPU) and phases, in the
    order a previous step leaves."""
    c = _constants(case)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    rand = lambda *s: torch.rand(*s, generator=gen, device=DEV)  # noqa: E731
    n = case["n"]
    if case["kind"] == "refcfg":
        grid, step, first, jitter = (case["side"],) * 3, 1.2, 4.0, 0.05
    else:
        w = case["w"] * (case["length"] if case.get("flow") == "splash" else 1)
        grid, step, first, jitter = (w, case["h"], case["d"]), S, 0.025, 0.005
        if case.get("flow") == "splash":
            jitter = 0.01
    total = grid[0] * grid[1] * grid[2]
    assert n <= total, case
    # which lattice sites hold a particle: the n smallest of E / weight
    site = torch.arange(total, device=DEV)
    if case.get("flow") == "splash":
        # a pool with waves, spray above it thinning out with height
        ph = rand(4) * 6.283
        fx, fz = (site // (grid[1] * grid[2])) / grid[0], (site % grid[2]) / grid[2]
        fy = ((site // grid[2]) % grid[1]) / grid[1]
        fill = 0.55 * n / total
        top = fill * (1.0 + 0.5 * torch.sin(6.283 * fx + ph[0]) * torch.cos(6.283 * fz + ph[1])
                      + 0.3 * torch.sin(18.85 * fx + ph[2]) + 0.2 * torch.cos(12.57 * fz + ph[3]))
        weight = torch.where(fy < top, torch.full_like(fy, 50.0), torch.exp(-(fy - top) / 0.3) + 0.02)
        score = -torch.log(rand(total) + 1e-12) / weight
        site = torch.sort(torch.topk(score, n, largest=False, sorted=False).indices).values
    elif n < total:
        site = torch.sort(torch.topk(rand(total), n, largest=False, sorted=False).indices).values
    ijk = torch.stack([site // (grid[1] * grid[2]), (site // grid[2]) % grid[1], site % grid[2]], 1).float()
    x = torch.ones(n, 4, device=DEV)
    x[:, :3] = first + step * ijk + (rand(n, 3) * 2.0 - 1.0) * jitter
    for a in range(3):
        x[:, a].clamp_(c["bmin"][a] + 0.001, c["bmax"][a] - 0.001)
    # a smooth velocity field (a few swirling modes) and a little noise
    amp = {"splash": 1.5}.get(case.get("flow"), 0.3) * (c["cell"] / CELL if case["kind"] == "refcfg" else 1.0)
    v = torch.zeros(n, 4, device=DEV)
    size = torch.tensor([c["bmax"][a] - c["bmin"][a] for a in range(3)], device=DEV)
    u = x[:, :3] / size * 6.283
    for a in range(3):
        for _ in range(3):
            k = torch.floor(rand(3) * 3.0) + 1.0
            v[:, a] += amp * (rand(1) * 2.0 - 1.0) * torch.sin((u * k).sum(1) + rand(1) * 6.283)
        v[:, a] += 0.05 * amp * torch.randn(n, generator=gen, device=DEV)
    f = torch.zeros(n, 4, device=DEV)
    f[:, :3] = 0.005 * torch.randn(n, 3, generator=gen, device=DEV)
    phase = torch.zeros(n, dtype=torch.int32, device=DEV)
    if case.get("solids"):
        # solid grains: the particles inside random spheres of two diameters
        side = 8.0 * 0.025
        cell = torch.floor(x[:, :3] / side).long()
        lin = (cell[:, 0] * 2048 + cell[:, 1]) * 2048 + cell[:, 2]
        mix = (lin * 2654435761 + int(seed) * 40503) % 1000003
        mix = (mix * 48271) % 1000003
        near = ((x[:, :3] / side - cell - 0.5) ** 2).sum(1) < 0.25
        phase = (near & (mix.double() < 1000003 * min(1.0, case["solids"] / 0.52))).int()
    # sorted by cell; with phases (which a program uploads once, and which follow
    # their particles) by the cell of the coming step, whose order they keep
    at = _predict32(c, x[:, :3], v[:, :3], f[:, :3]) if case.get("solids") else x
    o = torch.sort(_morton(_cells(c, at)), stable=True).indices
    return x[o].contiguous(), v[o].contiguous(), f[o].contiguous(), phase[o].contiguous()


class _DeviceArray:
    """A device buffer of a context as torch sees it (no copy).  A tensor holds on to
    the object it was made from, and so to the context whose memory it shows."""

    def __init__(self, ctx, ptr, n):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": (n, 4), "typestr": "<f4", "data": (int(ptr), False), "version": 2}


def _buffers(ctx):
    b = ctx.buffers()
    return {k: torch.as_tensor(_DeviceArray(ctx, getattr(b, a), b.num_particles), device=DEV)
            for k, a in (("x", "positions4"), ("p", "predicted_positions4"), ("v", "velocities4"), ("c", "colors4"),
                         ("f", "external_forces4"))}


# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "batch":
        # the case gives the scenes' sizes and boxes, the seed their particles and relaxation
        scenes = uneven_dam_breaks(F.config_path("dam_break_32k"), case["scenes"], seed=case["scenes"],
                                   lo=case["lo"], hi=case["hi"])
        rng = np.random.default_rng(seed)
        for k, p in enumerate(scenes):
            p.box_seed_lo = (seed * 1009 + k) & 0xFFFFFFFF
            p.relaxation = float(rng.uniform(300.0, 900.0))
        batch = F.capi.Batch(scenes)
        return {"kind": "batch", "batch": batch, "frames": case["frames"]}
    p = _params(case)
    x, v, f, phase = _state(case, seed)
    state = {"kind": case["kind"], "start": (x, v, f), "params": p}
    if case["kind"] == "noalloc":
        state["arrays"] = [x.clone(), x.clone(), v.clone(), torch.ones_like(x), f.clone()]
        return state
    ctx = F.Context(p, case["n"])
    ctx.add_particles(x.cpu().numpy(), v.cpu().numpy())
    state["ctx"] = ctx
    if case["kind"] == "adjoint":
        rng = np.random.default_rng(seed)
        host = {"positions": x.cpu().numpy(), "velocities": v.cpu().numpy(), "external_forces": f.cpu().numpy()}
        if case.get("solids"):
            host["phases"] = phase.cpu().numpy().astype(np.uint32)
        state.update(host=host, frames=case["frames"], target=_target(host["positions"], rng), start=None)
        return state
    if case.get("solids"):
        ctx.upload("phases", phase.cpu().numpy().astype(np.uint32))
    ctx.upload("external_forces", f.cpu().numpy())
    return state


def _target(x0, rng):
    """Where the loss wants the particles: the start spread out by 2 % about its
    middle, with a little noise."""
    x = x0[:, :3].astype(np.float64)
    return x + 0.02 * (x - x.mean(0)) + rng.normal(0.0, 0.005, x.shape)


def run(state):
    kind = state["kind"]
    if kind == "batch":
        b = state["batch"]
        b.step(state["frames"])
        return {"x": np.concatenate([b.download(s, "positions") for s in range(b.num_scenes)])}
    if kind == "noalloc":
        x, p, v, c, f = state["arrays"]
        for a, s in zip((x, v, f), state["start"]):
            a.copy_(s)
        rc = F.capi.lib().pbd_compute_noalloc(
            ctypes.byref(state["params"]), x.shape[0], x.data_ptr(), p.data_ptr(), v.data_ptr(), c.data_ptr(),
            f.data_ptr(), torch.cuda.current_stream().cuda_stream)
        F.capi.check(rc, "pbd_compute_noalloc")
        return {"x": x, "v": v, "f": f, "c": c}
    ctx = state["ctx"]
    if kind == "adjoint":
        n = ctx.n
        for k, a in state["host"].items():
            ctx.upload(k, a)
        ctx.adj_forward(state["frames"], 1)
        ids = ctx.adj_ids()
        xT = ctx.download("positions")
        gx = np.zeros((n, 4), np.float32)
        gx[:, :3] = (2.0 / n) * (xT[:, :3] - state["target"][ids])
        g = ctx.adj_backward(gx, None, x0=False)
        x = np.empty((n, 3), np.float32)
        x[ids] = xT[:, :3]
        return {"x": x, "v0": g["v0"], "rho0": g["rho0"], "eps": g["eps"]}
    # frame, refcfg: the context is idle here (the last pass waited for it); its
    # buffers are read and written by torch's stream between the steps
    b = _buffers(ctx)
    for k, s in zip(("x", "v", "f"), state["start"]):
        b[k].copy_(s)
    torch.cuda.current_stream().synchronize()
    ctx.step(1, graph=True)
    ctx.sync()
    return {k: b[k] for k in ("x", "v", "f", "c")}


def work(case):
    """State in (x, v, f) and out (x, p*, v, colour, f) once per substep; per
    iteration and particle about 33 pairs of 20 (lambda) and 35 (delta-p, contact)
    operations, then 60 for vorticity and XSPH.  The adjoint: a recorded forward, its
    recomputation and a reverse of twice the work."""
    if case["kind"] == "batch":
        n = case["scenes"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        return {"bytes": n * (128 * case["frames"] + 16), "flops": n * case["frames"] * 33 * 280}
    n = case["n"]
    if case["kind"] == "refcfg":  # 124 cells of 1/1.2^3 particles, one iteration
        return {"bytes": 128 * n, "flops": n * 71 * 130}
    if case["kind"] == "adjoint":
        sub = 2 * case["frames"]
        return {"bytes": n * (3 * 128 * sub + 16 * 5), "flops": n * sub * 33 * 280 * 4}
    pairs = 33 if case["flow"] == "column" else 20
    return {"bytes": 128 * n, "flops": n * pairs * 280}


# ---------------------------------------------------------------------------
# The step in 64 bits, in plain torch.
def _columns(c, ijk, lin, cum):
    """Candidate ranges of the stencil: per (dx, dy) the z cells -kw..kw of every
    particle as one range of the cell-sorted order (start, count)."""
    kw, dims = c["kw"], c["dims"]
    for dx in range(-kw, kw + 1):
        for dy in range(-kw, kw + 1):
            X, Y = ijk[:, 0] + dx, ijk[:, 1] + dy
            ok = (X >= 0) & (X < dims[0]) & (Y >= 0) & (Y < dims[1])
            row = (X.clamp(0, dims[0] - 1) * dims[1] + Y.clamp(0, dims[1] - 1)) * dims[2]
            a = cum[row + (ijk[:, 2] - kw).clamp(min=0)]
            b = cum[row + (ijk[:, 2] + kw).clamp(max=dims[2] - 1) + 1]
            yield a, torch.where(ok, b - a, torch.zeros_like(a))


def _pairs(c, ijk, lin, cum, x, radius):
    """All ordered candidate pairs (i, j), i != j, nearer than radius."""
    n, found = x.shape[0], []
    for a, cnt in _columns(c, ijk, lin, cum):
        i = torch.repeat_interleave(torch.arange(n, device=x.device), cnt)
        first = torch.cumsum(cnt, 0) - cnt
        j = torch.arange(i.shape[0], device=x.device) - first[i] + a[i]
        d = x[i] - x[j]
        m = ((d * d).sum(1) < radius * radius) & (i != j)
        found.append((i[m], j[m]))
    return torch.cat([p[0] for p in found]), torch.cat([p[1] for p in found])


def _add(n, i, t):
    out = torch.zeros((n,) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
    return out.index_add(0, i, t)


def _step64(c, x, v, f, phase, rho0, eps):
    """One substep: (x, v, f, colour) and the permutation to the step's order, all in
    that order.  x, v, f: n x 3 in 64 bits."""
    dt = float(np.float32(c["dt"]))
    # predict: the values are those of float32 arithmetic, the derivatives the formula's
    g = torch.tensor([0.0, c["gravity"] * dt, 0.0], dtype=x.dtype, device=x.device)
    p = x + (v + g + f * dt) * dt
    lo = torch.tensor(c["bmin"], dtype=x.dtype, device=x.device) + 0.001
    hi = torch.tensor(c["bmax"], dtype=x.dtype, device=x.device) - 0.001
    p32 = _predict32(c, x.detach().float(), v.detach().float(), f.detach().float())
    clamped = (p.detach() < lo - 0.001) | (p.detach() > hi + 0.001)
    p = torch.where(clamped, p32.to(x.dtype), p + (p32.to(x.dtype) - p).detach())
    ijk = _cells(c, p32)
    lin = (ijk[:, 0] * c["dims"][1] + ijk[:, 1]) * c["dims"][2] + ijk[:, 2]
    perm = torch.sort(lin, stable=True).indices
    ijk, lin = ijk[perm], lin[perm]
    counts = torch.bincount(lin, minlength=c["dims"][0] * c["dims"][1] * c["dims"][2])
    cum = torch.cat([torch.zeros(1, dtype=torch.long, device=x.device), torch.cumsum(counts, 0)])
    q, qx, ph = p[perm], x[perm], phase[perm].bool()
    n, text = x.shape[0], c["variant"] == 1
    fluid = ~ph
    hp, hs = c["hp"], c["hs"]
    if text:
        wc, gc = 315.0 / (64.0 * math.pi * hp ** 9), -45.0 / (math.pi * hs ** 6)
        w0, ks, vol = 315.0 / (64.0 * math.pi * hp ** 3), c["k_scorr"] * hs * hs, 1.0 / rho0
        w_dq = wc * (hp * hp - c["dq"] ** 2) ** 3
    else:
        wc, gc = 315.0 / (0.001 + 64.0 * math.pi * hp ** 9), 15.0 / (math.pi * hs ** 6)
        w0, ks, vol = 0.0, c["k_scorr"], 1.0
        w_dq = wc * (hp * hp - c["dq"] ** 2) ** 6

    def geometry(i, j):
        d = q[i] - q[j]
        r2 = (d * d).sum(1)
        r = torch.sqrt(torch.clamp(r2, min=1e-30))
        if text:
            w = torch.clamp(hp * hp - r2, min=0.0) ** 3
            hr = torch.clamp(hs - r, min=0.0)
            return d, r, w, hr * hr / r, hr ** 4
        w = torch.where((r > 0.001) & (r < hp - 0.001), (hp * hp - r2) ** 6, torch.zeros_like(r))
        hr = torch.where((r > 1e-4) & (hs - r > 1e-4), hs - r, torch.zeros_like(r))
        return d, r, w, hr * hr / r, hr ** 4

    radius = max(hp, hs, c["diameter"])
    for _ in range(c["iters"]):
        i, j = _pairs(c, ijk, lin, cum, q.detach(), radius)
        d, r, w, gr, hr4 = geometry(i, j)
        both = (fluid[i] & fluid[j]).to(x.dtype)
        wf = fluid[j].to(x.dtype)
        dens = wc * _add(n, i, w * wf) + w0
        G2 = gc * gc * (_add(n, i, d * (gr * wf)[:, None]) ** 2).sum(1)
        B2 = gc * gc * _add(n, i, hr4 * wf)
        lam = -(dens / rho0 - 1.0) / ((G2 + B2) / (rho0 * rho0 if text else rho0) + eps)
        lam = torch.where(ph, torch.zeros_like(lam), lam)
        sc = -ks * (wc * w / w_dq) ** c["n_scorr"]
        dp = gc / rho0 * _add(n, i, d * ((lam[i] + lam[j] + sc) * gr * both)[:, None])
        ov = torch.clamp(c["diameter"] - r, min=0.0)
        near = (ijk[i] - ijk[j]).abs().max(1).values <= 1  # contacts: the 27 cells
        ov = torch.where(near & (r > 1e-5), ov, torch.zeros_like(ov))
        push = _add(n, i, d * (0.5 * (1.0 - c["stiffness"]) * ov / r)[:, None])
        new = q + push
        if c["mu_s"] > 0.0:
            m = torch.nonzero((ov > 0.0) & (ph[i] | ph[j])).squeeze(1)
            a, b, nrm, depth = i[m], j[m], d[m] / r[m, None], ov[m]
            u = (q[a] - qx[a]) - (q[b] - qx[b])
            t = u - (u * nrm).sum(1, keepdim=True) * nrm
            tl = torch.sqrt(torch.clamp((t * t).sum(1), min=1e-40))
            s = torch.where(tl < c["mu_s"] * depth, torch.ones_like(tl), torch.clamp(c["mu_k"] * depth / tl, max=1.0))
            new = new - _add(n, a, 0.5 * s[:, None] * t)
        if text:
            off = torch.minimum(torch.maximum(new + dp, lo), hi)
            q = off
        else:
            q = new - dp
        qx = qx + push
    vel = (q - qx) / dt
    i, j = _pairs(c, ijk, lin, cum, q.detach(), radius)
    both = fluid[i] & fluid[j]
    i, j = i[both], j[both]
    d, r, w, gr, _ = geometry(i, j)
    dv = vel[j] - vel[i]
    om = _add(n, i, torch.linalg.cross(dv, d * gr[:, None])) * (-gc * vol if text else gc)
    vo = vel + c["c_visc"] * wc * vol * _add(n, i, dv * w[:, None])
    if text:
        ol = torch.sqrt(torch.clamp((om * om).sum(1), min=1e-60))
        e = gc * _add(n, i, d * ((ol[j] - ol[i]) * gr)[:, None])
        el = torch.sqrt(torch.clamp((e * e).sum(1, keepdim=True), min=1e-60))
        force = c["e_vort"] * torch.linalg.cross(e / el, om)
    else:
        force = None  # component quotients over differences of coordinates: unbounded in them
    cnt = sum(k for _, k in _columns(c, ijk, lin, cum)) - 1
    col = torch.clamp(cnt, max=c["cap"]).to(x.dtype) / c["cap"]
    o = torch.sort(_morton(ijk), stable=True).indices
    return q[o], vo[o], None if force is None else force[o], col[o], perm[o]


def exact(case, seed):
    # a batch's outputs stand several substeps on: their order follows cells that
    # rounding decides, and past 1.2M particles the pairs take too long here
    if case["kind"] == "batch" or case["n"] > 1200000:
        return None
    c = _constants(case)
    x, v, f, phase = _state(case, seed)
    x64, v64, f64 = (t[:, :3].double() for t in (x, v, f))
    if case["kind"] != "adjoint":
        q, vo, force, col, _ = _step64(c, x64, v64, f64, phase, c["rho0"], c["eps"])
        n = q.shape[0]
        one, zero = torch.ones(n, 1, device=q.device, dtype=q.dtype), torch.zeros(n, 1, device=q.device, dtype=q.dtype)
        return {"x": torch.cat([q, one], 1), "v": torch.cat([vo, zero], 1),
                "f": None if force is None else torch.cat([force, zero], 1),
                "c": torch.cat([col[:, None].expand(n, 3), one], 1)}
    target = torch.from_numpy(_target(x.cpu().numpy(), np.random.default_rng(seed))).to(DEV)
    v0 = v64.clone().requires_grad_()
    rho0 = torch.tensor(c["rho0"], dtype=torch.float64, device=DEV, requires_grad=True)
    eps = torch.tensor(c["eps"], dtype=torch.float64, device=DEV, requires_grad=True)
    at = torch.arange(case["n"], device=DEV)
    xs, vs, fs, ph = x64, v0, f64, phase
    for _ in range(2 * case["frames"]):
        xs, vs, fs, _, o = _step64(c, xs, vs, fs, ph, rho0, eps)
        at, ph = at[o], ph[o]
    loss = ((xs - target[at]) ** 2).sum() / case["n"]
    gv, gr, ge = torch.autograd.grad(loss, [v0, rho0, eps])
    out = torch.empty_like(x64)
    out[at] = xs.detach()
    return {"x": out, "v0": gv, "rho0": float(gr), "eps": float(ge)}

"""The work this framework is measured on, through its public entry points.

A case is one burst of a simulation as a user's program runs it: a number of
whole time steps on a state that lives on the GPU, then the state back in the
host's buffers (the reference's loop writes a layer every so many steps); or a
differentiable run, forward and backward.  The sizes are those of the
repository's configurations (the 6.9k-particle dam break, the piston flume at
its stated spacing and at 1M particles, the 6.6M-particle 3D dam break, the
134k-particle wave tank, the 3D piston basin) and others of the same ranges.

Flows start in motion (a standing wave in the flumes, the straining flow of a
collapsing column in the dam breaks, a seeded jitter of the positions), as a
run restarted from a dump does.  Most cases go on from pass to pass; the
short 2D dam break uploads its initial state again in every pass, as a
parameter study does.

An FP32 context keeps velocities, densities and pressures in FP32 and widens
them on download: its outputs are stored as float32 here (positions are FP64 in
both precisions).
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P
from sph2d_amd.adjoint import DifferentiableRun, PistonGauges


def listed():
    return [
        # the smallest run: the 2D dam break of 6,923 particles, FP64, where launches and latency count
        {"name": "dam2d_7k_f64", "kind": "dam2d", "delta": 0.01, "fp64": True, "steps": 200},
        # the piston flume at its stated spacing, dynamic CFL time step
        {"name": "flume_188k_f32", "kind": "flume", "delta": 0.0075, "length": 20.0, "depth": 0.5, "fp64": False,
         "steps": 32},
        # the headline workload, in both precisions
        {"name": "flume_1m_f32", "kind": "flume", "delta": 0.0031623, "length": 20.0, "depth": 0.5, "fp64": False,
         "steps": 50},
        {"name": "flume_1m_f64", "kind": "flume", "delta": 0.0031623, "length": 20.0, "depth": 0.5, "fp64": True,
         "steps": 50},
        # summation density in 2D
        {"name": "sum2d_135k_f32", "kind": "sum2d", "delta": 0.002, "fp64": False, "steps": 30},
        # the options outside the cubic configuration: Wendland kernels, delta-SPH, artificial pressure
        {"name": "wendland_188k_f64", "kind": "wendland", "delta": 0.0075, "length": 20.0, "depth": 0.5, "fp64": True,
         "steps": 32},
        # the 3D dam break (summation density renormalised every 30th step), coarse in FP64 and at its stated spacing
        {"name": "dam3d_556k_f64", "kind": "dam3d", "delta": 0.0065, "fp64": True, "steps": 25},
        {"name": "dam3d_6m6_f32", "kind": "dam3d", "delta": 0.0025, "fp64": False, "steps": 16},
        # the differentiable 2D wave tank: forward with gauges and reverse pass
        {"name": "tank_134k_adjoint_f64", "kind": "tank", "delta": 0.005, "length": 8.0, "fp64": True, "steps": 60,
         "every": 20},
        # the differentiable 3D basin through torch.autograd, FP32 steps
        {"name": "basin_1m_adjoint_f32", "kind": "basin", "delta": 0.02, "length": 6.0, "fp64": False, "steps": 12,
         "every": 6},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: a kind, a particle count over its range, precision and number of steps."""
    kind = rng.choice(["dam2d", "flume", "flume", "sum2d", "wendland", "dam3d", "tank", "basin"])
    fp64 = rng.random() < 0.5
    if kind == "dam2d":
        n = _log(rng, 3000, 3e5)
        return {"kind": kind, "delta": round(math.sqrt(0.5 / n) * 1.15, 6), "fp64": True, "steps": rng.randint(40, 200)}
    if kind in ("flume", "wendland"):
        length, depth = round(rng.uniform(6.0, 20.0), 2), round(rng.uniform(0.3, 0.5), 3)
        delta = round(math.sqrt(length * depth / _log(rng, 4000, 1e6 if kind == "flume" else 4e5)), 6)
        # a coarse FP32 run takes fewer steps between layers: its time step is longer
        most = 50 if fp64 else max(6, min(50, int(0.25 / delta)))
        return {"kind": kind, "delta": delta, "length": length, "depth": depth, "fp64": fp64,
                "steps": rng.randint(most // 2, most)}
    if kind == "sum2d":
        delta = round(math.sqrt(0.5 / _log(rng, 2e4, 5e5)), 6)
        most = 30 if fp64 else max(6, min(30, int(0.06 / delta)))
        return {"kind": kind, "delta": delta, "fp64": fp64, "steps": rng.randint(most // 2, most)}
    if kind == "dam3d":
        delta = round(0.0025 * (4.6e6 / _log(rng, 3e4, 2e6)) ** (1 / 3), 6)
        most = 25 if fp64 else max(4, min(16, int(0.04 / delta)))
        return {"kind": kind, "delta": delta, "fp64": fp64, "steps": rng.randint(max(most // 2, 3), most)}
    if kind == "tank":
        length = round(rng.uniform(3.0, 8.0), 2)
        return {"kind": kind, "delta": round(math.sqrt(length * 0.4 / _log(rng, 5000, 1.3e5)), 6), "length": length,
                "fp64": True, "steps": rng.randint(15, 60), "every": rng.randint(5, 30)}
    length = round(rng.uniform(2.0, 6.0), 2)
    return {"kind": "basin", "delta": round((length * 2.0 * 0.5 / _log(rng, 4e4, 7e5)) ** (1 / 3), 6),
            "length": length, "fp64": fp64, "steps": rng.randint(4, 12), "every": rng.randint(2, 8)}


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=2)
def _layout(key):
    c = dict(key)
    kind, delta = c["kind"], c["delta"]
    if kind == "dam2d":
        return G.dam_break(delta=delta, jitter=0.0, dt=5e-5 * delta / 0.01)
    if kind == "sum2d":
        lay = G.dam_break(delta=delta, jitter=0.0, dt=5e-5 * delta / 0.01, density_treatment=P.DENSITY_SUMMATION)
        lay.params.consistency_treatment = P.CONSISTENCY_FIX
        return lay
    if kind == "flume":
        return G.piston_tank(delta=delta, length=c["length"], depth=c["depth"])
    if kind == "wendland":
        lay = G.piston_tank(delta=delta, length=c["length"], depth=c["depth"])
        prm = lay.params
        prm.density_skf = prm.intf_skf = prm.artificial_viscosity_skf = prm.average_velocity_skf = P.SKF_WENDLAND
        prm.artificial_pressure_skf = P.SKF_WENDLAND
        prm.density_treatment = P.DENSITY_CONTINUITY_DELTA
        prm.density_delta_sph_coef = 0.1
        prm.artificial_pressure, prm.artificial_pressure_coef, prm.artificial_pressure_index = True, 0.2, 4.0
        P.fill_in_computing_params(prm)
        P.post_fill_in_model_params(prm)
        return lay
    if kind == "dam3d":
        lay = G.dam_break_3d(delta=delta, box=(1.6, 0.8, 0.6), column=(0.4, 0.3, 0.6), jitter=0.0)
        lay.params.density_normalization, lay.params.density_normalization_every = 1, 30
        lay.params.consistency_treatment = P.CONSISTENCY_FIX
        return lay
    if kind == "tank":
        return G.adjoint_tank(delta=delta, length=c["length"])
    return G.piston_basin_3d(delta=delta, length=c["length"])


def _inputs(case, seed):
    """Layout and the initial state: positions with a seeded jitter, the fluid in motion."""
    lay = _layout(tuple(sorted((k, v) for k, v in case.items() if k in ("kind", "delta", "length", "depth"))))
    prm, nf = lay.params, lay.params.nfluid
    rng = np.random.default_rng(seed)
    r, v = lay.r.copy(), np.zeros_like(lay.r)
    jitter = (0.002 if case["kind"] in ("sum2d", "dam3d") else 0.01) * prm.delta
    r[:nf] += rng.uniform(-jitter, jitter, size=(nf, prm.dim))
    x, y = r[:nf, 0], r[:nf, 1]
    if case["kind"] in ("dam2d", "sum2d", "dam3d"):
        s = rng.uniform(0.8, 1.2)  # the straining flow of the collapse, v = s (x, -y)
        v[:nf, 0], v[:nf, 1] = s * x, -s * y
    else:
        length, depth = float(x.max() + x.min()), float(y.max())
        for m in range(1, 6):  # standing waves between the end walls at the instant the surface is level
            k, amp = m * math.pi / length, 0.2 * rng.uniform(0.3, 1.0) / m
            v[:nf, 0] += amp * np.sin(k * x) * np.cosh(k * y) / math.cosh(k * depth)
            v[:nf, 1] -= amp * np.cos(k * x) * np.sinh(k * y) / math.cosh(k * depth)
    return lay, r, v, rng


def _gauges(case, prm):
    """Gauges within the distance that sound travels in the run, so that every one sees the piston."""
    reach = max(prm.eos_c * case["steps"] * prm.dt, 8 * prm.delta)
    if case["kind"] == "tank":
        xs, zs = [2 * prm.delta + reach * (i + 1) / 5 for i in range(4)], None
    else:
        xs = [2 * prm.delta + reach * (i + 1) / 5 for i in range(4) for _ in range(4)]
        zs = [z for _ in range(4) for z in (0.25, 0.75, 1.25, 1.75)]
    return xs, zs, 3 * prm.delta, prm.delta / 4, prm.depth


def _out_buffers(prm, fp64):
    """The host arrays a program keeps for the layers it reads back, pinned."""
    n, d = prm.ntotal, prm.dim

    def pinned(shape, dtype=torch.float64):
        return torch.empty(shape, dtype=dtype, pin_memory=torch.cuda.is_available())

    out = {"r": pinned((n, d)), "v": pinned((n, d)), "rho": pinned(n), "p": pinned(n),
           "itype": pinned(n, torch.int32)}
    narrow = None if fp64 else {f: torch.empty(out[f].shape, dtype=torch.float32) for f in ("v", "rho", "p")}
    return out, narrow


def prepare(case, seed):
    lay, r, v, rng = _inputs(case, seed)
    prm = lay.params
    sim = H.HipStep(prm, precision=H.FP64 if case["fp64"] else H.FP32)
    state = {"case": case, "sim": sim}
    init = {"r": r, "v": v, "rho": lay.rho, "itype": lay.itype}
    if case["kind"] in ("tank", "basin"):
        xs, zs, radius, tau, y_ref = _gauges(case, prm)
        spec = H.gauge_spec(xs, radius=radius, tau=tau, y_ref=y_ref, zs=zs)
        state["run"] = DifferentiableRun(sim, init, case["steps"], case["every"], spec, prm.piston_omega)
        # coefficients of this seed; an FP32 program holds them in float32
        dtype = torch.float64 if case["fp64"] else torch.float32
        state["a"], state["b"], state["target"] = (torch.tensor(t).to(dtype) for t in _coefficients(case, prm, rng))
        return state
    state["out"], state["narrow"] = _out_buffers(prm, case["fp64"])
    if case["kind"] == "dam2d":
        state["init"] = init
    else:
        sim.upload(**init)
    return state


def _coefficients(case, prm, rng):
    """Piston coefficients a, b and the target gauge elevations of the loss."""
    scale = 0.005 if case["kind"] == "tank" else 0.01
    nc, ng = len(prm.piston_a), 4 if case["kind"] == "tank" else 16
    return (rng.normal(0, scale, nc), rng.normal(0, scale, nc),
            prm.depth + rng.normal(0, 0.02, size=(case["steps"], ng)))


def run(state):
    case, sim = state["case"], state["sim"]
    if case["kind"] == "tank":
        # the loss's gradients with respect to the coefficients and the initial state
        eta = state["run"].forward(state["a"].numpy(), state["b"].numpy())
        grads = state["run"].backward(2.0 * (eta - state["target"].numpy()), len(state["a"]))
        return {"eta": eta, **grads}
    if case["kind"] == "basin":
        a, b = state["a"].clone().requires_grad_(True), state["b"].clone().requires_grad_(True)
        eta = PistonGauges.apply(a, b, state["run"])
        ((eta - state["target"].double()) ** 2).sum().backward()
        return {"eta": eta.detach(), "a": a.grad, "b": b.grad}
    if case["kind"] == "dam2d":
        sim.upload(**state["init"])
    sim.step(case["steps"])
    out = state["out"]
    dp = ctypes.POINTER(ctypes.c_double)
    status = sim.L.rrsph_hip_download(sim.ctx, 31, *(ctypes.cast(out[f].data_ptr(), dp) for f in ("r", "v", "rho", "p")),
                                      ctypes.cast(out["itype"].data_ptr(), ctypes.POINTER(ctypes.c_int32)))
    if status:
        raise H.RrsphError(status, sim.L.rrsph_hip_last_error(sim.ctx).decode())
    if state["narrow"] is None:
        return out
    for f, t in state["narrow"].items():
        t.copy_(out[f])
    return {**out, **state["narrow"]}


# ---------------------------------------------------------------- work
def work(case):
    """Per step: position, velocity and density, and the last acceleration, each read and written once; a pair's
    arithmetic once for each particle of it.  Reverse steps read the state and read and write its adjoint."""
    prm = _layout(tuple(sorted((k, v) for k, v in case.items() if k in ("kind", "delta", "length", "depth")))).params
    n, d, w = prm.ntotal, prm.dim, 8 if case["fp64"] else 4
    state = 8 * d + 2 * w * (d + 1)
    pairs, flops = (20, 70) if d == 2 else (80, 85)
    if case["kind"] in ("sum2d", "dam3d"):
        flops += 20
    fwd, fl = 2 * state, pairs * flops
    if case["kind"] in ("tank", "basin"):
        fwd, fl = fwd + state + 2 * 8 * (3 * d + 2), fl + pairs * 4 * flops
    return {"bytes": float(n) * case["steps"] * fwd, "flops": float(n) * case["steps"] * fl}


# ---------------------------------------------------------------- the same in 64 bits with torch
def _pairs(prm, r):
    """Ordered pairs (j, i) with |r_i - r_j|^2 < (k h)^2, from a sort by cell of side k h."""
    d, cell, n = prm.dim, prm.cell_scale_k * prm.hsml, len(r)
    lo = torch.tensor([prm.x_mingeom, prm.y_mingeom, prm.z_mingeom][:d], dtype=r.dtype, device=r.device)
    cells = ((r - lo) / cell).floor().long() + 1
    dims = cells.max(0).values + 2
    key = cells[:, 0]
    for a in range(1, d):
        key = key * dims[a] + cells[:, a]
    order = torch.argsort(key)
    skey = key[order].contiguous()
    steps = [(dx,) for dx in (-1, 0, 1)] if d == 2 else [(dx, dy) for dx in (-1, 0, 1) for dy in (-1, 0, 1)]
    js, is_ = [], []
    for s in steps:
        base = key + s[0] * (dims[1] if d == 2 else dims[1] * dims[2])
        if d == 3:
            base = base + s[1] * dims[2]
        b, e = torch.searchsorted(skey, base - 1), torch.searchsorted(skey, base + 1, right=True)
        cnt = e - b
        j = torch.repeat_interleave(torch.arange(n, device=r.device), cnt)
        first = torch.repeat_interleave(b - (torch.cumsum(cnt, 0) - cnt), cnt)
        i = order[first + torch.arange(len(j), device=r.device)]
        keep = ((r[i] - r[j]).square().sum(1) < cell * cell) & (i != j)
        js.append(j[keep])
        is_.append(i[keep])
        del j, i, first, keep
    return torch.cat(js), torch.cat(is_)


def _kernel(prm, skf, dist):
    """W and its gradient's factor F (grad W = (r_i - r_j) F) of the cubic spline and the Wendland kernel."""
    h, pi = prm.hsml, math.pi
    q, t = dist / h, 2 - dist / h
    if skf == P.SKF_WENDLAND:
        f, s = 7 / (4 * pi * h * h), 0.5 * t
        return f * s**4 * (2 * q + 1), 2 * f / h / dist * (s**4 - (2 * q + 1) * s**3)
    f = 15 / (7 * pi * h * h) if prm.dim == 2 else 3 / (2 * pi * h**3)
    w = torch.where(q <= 1, f * (2 / 3 - q * q + 0.5 * q**3), f / 6 * t**3)
    return w, torch.where(q <= 1, f / h**2 * (-2 + 1.5 * q), -f / dist / h * 0.5 * t * t)


class _Flow:
    """One whole time step of the same method (predict, density, forces, whole step)."""

    def __init__(self, lay):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.prm, prm = lay.params, lay.params
        self.t = torch.from_numpy(lay.itype).to(dev)
        self.fluid, self.wall = (self.t > 0), (self.t < 0)
        idx = torch.arange(prm.ntotal, device=dev)
        self.paddle = (idx >= prm.nwm_particles_start) & (idx < prm.nwm_particles_end) & (idx >= prm.nfluid)
        self.dynamic = prm.dt_correction_method == P.DT_CORRECTION_DYNAMIC and prm.dt_dynamic_mode == 1

    def eos(self, rho):
        return self.prm.eos_c_sqr * self.prm.rho0 / 7 * ((rho / self.prm.rho0) ** 7 - 1)

    def piston(self, time, a, b, r):
        """Velocity of every particle of the Fourier piston (paddles across z in 3D)."""
        prm = self.prm
        segs = max(prm.piston_segments, 1)
        kw = torch.arange(1, len(a) // segs + 1, device=r.device, dtype=r.dtype) * prm.piston_omega
        vel = (kw * (a.view(segs, -1) * torch.cos(kw * time) - b.view(segs, -1) * torch.sin(kw * time))).sum(1)
        if segs == 1:
            return vel[0].expand(len(r))
        width = (prm.piston_seg_zmax - prm.piston_seg_zmin) / segs
        return vel[((r[:, 2].detach() - prm.piston_seg_zmin) / width).floor().long().clamp(0, segs - 1)]

    def step(self, r, v, rho, acc, drho, time, dt, k, a=None, b=None):
        prm, m, h = self.prm, self.prm.mass, self.prm.hsml
        summed = prm.density_treatment == P.DENSITY_SUMMATION
        j, i = _pairs(prm, r.detach())
        d = r[i] - r[j]
        d2 = d.square().sum(1)
        dist = d2.sqrt()
        w, f = _kernel(prm, prm.density_skf, dist)

        def gather(x):  # sum over the neighbours of each particle
            return torch.zeros((len(r),) + x.shape[1:], dtype=x.dtype, device=x.device).index_add(0, j, x)

        u = v + acc * (dt * 0.5)
        if summed:
            w0 = float(_kernel(prm, prm.density_skf, torch.zeros(1, dtype=r.dtype))[0])
            rh = m * w0 + gather(m * w)
            if prm.density_normalization and (k + 1) % prm.density_normalization_every == 0:
                rh = rh / (m / rho * w0 + gather(m / rho[i] * w))
            p = self.eos(rh)
            dr = torch.zeros_like(rho)
        else:
            rh, p = rho + drho * (dt * 0.5), self.eos(rho)
            pair = m * f * ((v[i] - v[j]) * d).sum(1)
            if prm.density_treatment == P.DENSITY_CONTINUITY_DELTA:
                c = 2 * prm.density_delta_sph_coef * h * prm.eos_c * m
                pair = pair + c * ((rho[i] - rho[j]) / rho[i]) * -f
            dr = gather(pair)
        pw = p / (rh * rh)
        coef = pw[i] + pw[j]
        if prm.artificial_pressure:
            wd = float(_kernel(prm, prm.artificial_pressure_skf, torch.full((1,), prm.delta, dtype=r.dtype))[0])
            tens = -prm.artificial_pressure_coef * torch.clamp(pw, max=0.0)
            coef = coef + (tens[i] + tens[j]) * (w / wd) ** prm.artificial_pressure_index
        du = u[i] - u[j]
        vr = (du * d).sum(1)
        mu = torch.where(vr < 0, h * vr / (d2 + (float(np.float32(0.1)) * h) ** 2), torch.zeros_like(vr))
        irho = 1.0 / (rh[i] + rh[j])
        coef = coef + (prm.artificial_bulk_visc * mu - prm.artificial_shear_visc * prm.eos_sound_vel) * mu * 2 * irho
        force = (m * f * coef)[:, None] * d
        rn = 2 * h / dist
        near = self.fluid[j] & self.wall[i] & (rn > 1)
        lj = torch.where(near, 5 * prm.g * prm.depth * (rn**12 - rn**4) / d2, torch.zeros_like(d2))
        an = gather(force - lj[:, None] * d)
        an = an - prm.g * torch.eye(prm.dim, dtype=r.dtype, device=r.device)[1]
        cw = torch.where(self.fluid[i], 2 * prm.average_velocity_coef * m * irho * w, torch.zeros_like(w))
        av = gather(cw[:, None] * du)
        if self.dynamic:
            top, most = float(an.square().sum(1).max().sqrt()), float(mu.abs().max())
            dt = prm.CFL_coef * min(math.sqrt(h / top), h / (prm.eos_c + most))
        vdt = dt * 0.5 if k == 0 else dt
        vn = torch.where(self.fluid[:, None], v + an * vdt + av, v)
        moving = self.fluid
        if prm.boundary_motion:
            moving = moving | self.wall
            vx = self.piston(time, a, b, r)
            vn = torch.where(self.paddle[:, None], torch.stack([vx] + [vx * 0] * (prm.dim - 1), 1), vn)
        rn_ = r + vn * dt * moving[:, None]
        return rn_, vn, rh if summed else rho + dr * vdt, an, dr, time + dt, dt, p

    def gauges(self, case, r):
        xs, zs, radius, tau, y_ref = _gauges(case, self.prm)
        y, out = r[self.fluid], []
        for g, x in enumerate(xs):
            s = (y[:, 0] - x) ** 2 + ((y[:, 2] - zs[g]) ** 2 if zs else 0.0)
            w = torch.clamp(1 - s / radius**2, min=0.0) ** 3
            out.append(y_ref + tau * torch.log((w * torch.exp((y[:, 1] - y_ref) / tau)).sum() / w.sum()))
        return torch.stack(out)


def exact(case, seed):
    lay, r, v, rng = _inputs(case, seed)
    prm = lay.params
    if prm.ntotal * case["steps"] * (1 if prm.dim == 2 else 6) > (2e7 if case["kind"] == "tank" else 9e7):
        return None
    if case["kind"] == "basin":
        return None
    flow = _Flow(lay)
    dev = flow.t.device
    r, v, rho = (torch.from_numpy(x).to(dev).clone() for x in (r, v, lay.rho))
    if case["kind"] == "tank":
        a, b, target = (torch.tensor(t, device=dev) for t in _coefficients(case, prm, rng))
        leaves = [x.requires_grad_(True) for x in (a, b, r, v, rho)]
    else:
        a, b = (torch.tensor(t, dtype=torch.float64, device=dev) for t in (prm.piston_a, prm.piston_b))
    s = (r, v, rho, torch.zeros_like(v), torch.zeros_like(rho))
    time, dt, etas, p = 0.0, prm.dt, [], None
    for k in range(case["steps"]):
        if case["kind"] == "tank":
            # each step is computed again in the backward pass
            *s, time, dt, p = checkpoint(flow.step, *s, time, dt, k, a, b, use_reentrant=False)
            etas.append(flow.gauges(case, s[0]))
        else:
            *s, time, dt, p = flow.step(*s, time, dt, k, a, b)
    if case["kind"] == "tank":
        eta = torch.stack(etas)
        grads = torch.autograd.grad(((eta - target) ** 2).sum(), leaves)
        return {"eta": eta.detach(), **dict(zip(("a", "b", "r", "v", "rho"), grads))}
    return {"r": s[0], "v": s[1], "rho": s[2], "p": p, "itype": None}

"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the public Python entry points (fwgpu.Solver,
fwgpu.Batch, fwcnn.Net), which are thin calls of the C ABI:

  flume    the reference's 1-D benchmark set-up: a few rows, periodic in y,
           WK_REG waves onto a planar beach, whole steps (fw_step)
  beach    the large-domain workload and its smaller relatives: a barred
           beach under directional JONSWAP waves (WK_DATA2D), three sponges,
           wetting and drying, breaking, whole steps
  member   one domain of an ensemble: slope and bumps, WK_REG waves
  shallow  the non-dispersive equations with a fixed step, friction and
           diffusion sponges and bottom friction
  routines one whole step through the per-routine entry points, in the order
           the Fortran drop-in's main loop calls them
  batch    an ensemble of uneven members advanced together (fw_batch)
  learned  a coarse run with the learned correction after every step
  train    one Adam step of the correction network on random crops
  predict  the network on host arrays (evaluation of a trained network)
  output   what a run does at an output interval: the budget of the domain
           and the output fields, brought to the host

A solver's pass is a few whole steps; it returns views of the resident state
(the arrays a run carries from step to step) and the clock.  The sea state is
developed from the start: random waves over the wet part of the domain, so
that limiters, breaking and the wet/dry front have work as in a real run.
"""
import ctypes as ct
import math
import os
import sys

import numpy as np
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(os.path.dirname(HERE), "funwave-tvd_amd"))

import fwcases  # noqa: E402
import fwcnn  # noqa: E402
import fwgpu  # noqa: E402
import fwlearn  # noqa: E402
import fwsetup  # noqa: E402

# the arrays a run carries from one step to the next
STATE = ("Eta", "U", "V", "HU", "HV", "Ubar", "Vbar", "H", "MASK", "AGE_BREAKING", "nu_break", "P", "Q")
OUTPUT = ("Eta", "U", "V", "MASK")
# words per cell and step that a whole step has to move: every field that
# crosses HBM when the intermediates of a stage stay on chip
STEP_WORDS = 93
# operations per cell and step: 3 stages of 14 limited reconstructions
# (about 50 each), the dispersion stencils (about 350) and the update with
# its source terms and two line solves (about 250)
STEP_FLOPS = 3 * (14 * 50 + 350 + 250)


def listed():
    return [
        # the reference's 1-D benchmark: the smallest call, bound by latency
        {"name": "flume_1024x4", "kind": "flume", "M": 1024, "N": 4, "prec": "sp", "steps": 10},
        # a small tank or a parameter study's domain
        {"name": "beach_96x72", "kind": "beach", "M": 96, "N": 72, "prec": "sp", "dx": 2.0, "steps": 10},
        # one ensemble member, no side a multiple of a tile
        {"name": "member_517x389", "kind": "member", "M": 517, "N": 389, "prec": "sp", "dx": 2.0, "steps": 5},
        # the headline workload
        {"name": "beach_2048x2048", "kind": "beach", "M": 2048, "N": 2048, "prec": "sp", "dx": 2.0, "steps": 2},
        # a production run in double precision, spacing no power of two
        {"name": "beach_1021x770_fp64", "kind": "beach", "M": 1021, "N": 770, "prec": "dp", "dx": 1.5, "steps": 2},
        # inundation without dispersion
        {"name": "shallow_777x601", "kind": "shallow", "M": 777, "N": 601, "prec": "sp", "dx": 2.0, "steps": 4},
        # the Fortran program with the drop-in routines
        {"name": "routines_512x384", "kind": "routines", "M": 512, "N": 384, "prec": "sp", "dx": 2.0, "steps": 1},
        # an ensemble in one launch per phase
        {"name": "batch_16", "kind": "batch", "members": 16, "M": 640, "N": 448, "prec": "sp", "steps": 4},
        # a learned coarse run
        {"name": "learned_700x468", "kind": "learned", "M": 700, "N": 468, "prec": "sp", "steps": 1},
        # the training loop's step at its default crop and batch
        {"name": "train_16x64x64", "kind": "train", "B": 16, "M": 64, "N": 64},
        # evaluation on a few held-out samples
        {"name": "predict_4x192x128", "kind": "predict", "B": 4, "M": 192, "N": 128},
        # an output interval
        {"name": "output_1024x768", "kind": "output", "M": 1024, "N": 768, "prec": "sp", "dx": 2.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flume", "beach", "beach", "member", "shallow", "routines", "batch", "learned", "train",
                       "predict", "output"])
    prec = rng.choice(["sp", "sp", "sp", "dp"])
    if kind == "flume":
        return {"kind": kind, "M": _log(rng, 160, 3000), "N": rng.randint(3, 8), "prec": prec, "steps": 10}
    if kind in ("beach", "member", "shallow", "routines", "output"):
        top = 1600 if prec == "sp" else 1100
        m, n = _log(rng, 80, top), _log(rng, 60, top)
        steps = 1 if kind == "routines" else max(1, min(10, int(2.5e6 / (m * n))))
        c = {"kind": kind, "M": m, "N": n, "prec": prec, "dx": rng.choice([2.0, 2.0, 1.5]), "steps": steps}
        if kind == "output":
            del c["steps"]
        return c
    if kind == "batch":
        return {"kind": kind, "members": rng.randint(3, 20), "M": _log(rng, 160, 640), "N": _log(rng, 120, 480),
                "prec": rng.choice(["sp", "sp", "dp"]), "steps": 3}
    if kind == "learned":
        return {"kind": kind, "M": rng.randint(256, 768), "N": rng.randint(128, 512), "prec": "sp", "steps": 1}
    if kind == "train":
        s = rng.randint(32, 96)
        return {"kind": kind, "B": rng.randint(2, 24), "M": s, "N": s}
    return {"kind": kind, "B": rng.randint(1, 8), "M": _log(rng, 48, 384), "N": _log(rng, 40, 256)}


# ---- inputs -----------------------------------------------------------------
def _flume(c, seed):
    """The 1-D beach; waves and toe placed in proportion to the length."""
    rng = np.random.default_rng(seed)
    m = c["M"]
    return fwcases.beach_1d(mglob=m, nglob=c["N"], xslp=0.39 * m, xc_wk=0.2 * m, sponge_west=0.1 * m,
                            amp=float(rng.uniform(0.3, 0.5)), period=float(rng.uniform(7.0, 9.0)))


def _beach(c, seed):
    """The barred beach at any size: the still-water depth follows the
    domain's length, so that its shore always lies inside the domain, and
    the waves follow the depth."""
    m, n, dx = c["M"], c["N"], c["dx"]
    lx = m * dx
    flat = min(20.0, 0.25 * lx / 20.0)
    case = fwcases.beach_2d(mglob=m, nglob=n, dx=dx, seed=2 * seed + 1, phase_seed=2 * seed + 2, flat_depth=flat,
                            slope=1.4 * flat / (0.27 * lx), shoal=(2400.0, None, 0.15 * flat, 150.0),
                            noise_std=0.01 * flat)
    case.spectrum["amp"] = case.spectrum["amp"] * (flat / 20.0)
    return case


def _member(c, seed):
    case = fwcases.member(seed, dx=c.get("dx", 2.0), mrange=(c["M"], c["M"]), nrange=(c["N"], c["N"]))
    case.params["AMP_WK"] = min(case.params["AMP_WK"], 0.6)
    return case


def _shallow(c, seed):
    case = _beach(c, seed)
    case.params.update({"DISPERSION": False, "DIRECT_SPONGE": False, "FRICTION_SPONGE": True,
                        "DIFFUSION_SPONGE": True, "CDsponge": 2.0, "Csp": 0.2, "Cd": 0.003,
                        "DT_fixed": fwlearn.stable_dt(case, cfl=0.4)})
    return case


def _island(c, seed):
    case = fwcases.island(seed, dx=4.0, mglob=c["M"], nglob=c["N"], h0=6.0, r_base=0.1 * 4.0 * min(c["M"], c["N"]))
    return fwlearn.with_fixed_dt(case, fwlearn.stable_dt(case, cfl=0.4))


CASE = {"flume": _flume, "beach": _beach, "member": _member, "shallow": _shallow, "routines": _beach,
        "learned": _island, "output": _beach}


def _sea(st, seed):
    """Random long-crested waves over the water deeper than an eighth of the
    domain's depth (the others are at rest), linear theory in shallow water:
    surface, velocities and the momentum the solver carries."""
    rng = np.random.default_rng(seed + 77)
    dep = st["Depth"].astype(np.float32)
    N, M = dep.shape
    flat = float(dep.max())
    x = (np.arange(M, dtype=np.float32) + 0.5) * st["DX"]
    y = (np.arange(N, dtype=np.float32) + 0.5) * st["DY"]
    K = 8
    lam = np.exp(rng.uniform(np.log(6.0), np.log(20.0), K)) * flat
    lam = np.maximum(lam, 12.0 * st["DX"])
    th = rng.uniform(-0.6, 0.6, K) if not st["PERIODIC"] else np.zeros(K)
    k = 2.0 * np.pi / lam
    a = 0.02 * flat * rng.uniform(0.5, 1.0, K) / math.sqrt(K)
    ph = rng.uniform(0.0, 2.0 * np.pi, K)
    ax, ay = np.outer(x, k * np.cos(th)) + ph, np.outer(y, k * np.sin(th))

    def field(w):  # sum_k w_k cos(ax + ay)
        w = w.astype(np.float32)
        return ((np.cos(ay).astype(np.float32) * w) @ np.cos(ax).astype(np.float32).T
                - (np.sin(ay).astype(np.float32) * w) @ np.sin(ax).astype(np.float32).T)

    ramp = np.clip((dep - 0.125 * flat) / (0.5 * flat), 0.0, 1.0)
    c = np.sqrt(9.81 / np.maximum(dep, 0.125 * flat))
    rdt = st["Depth"].dtype
    wet = ramp > 0
    eta = np.where(wet, ramp * field(a), st["Eta"])
    u, v = ramp * c * field(a * np.cos(th)), ramp * c * field(a * np.sin(th))
    h = np.where(wet, eta + dep, st["H"])
    for name, val in (("Eta", eta), ("U", u), ("V", v), ("H", h), ("HU", h * u), ("HV", h * v), ("Ubar", h * u),
                      ("Vbar", h * v)):
        st[name] = val.astype(rdt)
    return st


def _solver(c, seed):
    case = CASE[c["kind"]](c, seed)
    return fwgpu.Solver(_sea(fwsetup.build_state(case, c["prec"]), seed), c["prec"])


def _members(c, seed):
    """Uneven members: sides from half to one and a half times the mean."""
    rng = np.random.default_rng(seed)
    out = []
    rows = np.random.default_rng(c["M"] * 1000 + c["N"])  # the sizes belong to the case, not to the seed
    for k in range(c["members"]):
        m, n = int(rows.integers(c["M"] // 2, 3 * c["M"] // 2)), int(rows.integers(c["N"] // 2, 3 * c["N"] // 2))
        case = _member({"M": m, "N": n}, int(rng.integers(1 << 20)))
        case = fwlearn.with_fixed_dt(case, fwlearn.stable_dt(case, cfl=0.35))
        out.append(fwgpu.Solver(_sea(fwsetup.build_state(case, c["prec"]), seed + k), c["prec"]))
    return out


def _net_data(c, seed):
    """Samples as the network meets them: smooth scaled surfaces and
    velocities, depth, a wet mask with some land; targets of a few units."""
    rng = np.random.default_rng(seed)
    B, H, W = c["B"], c["N"], c["M"]
    yy, xx = np.meshgrid(np.arange(H), np.arange(W), indexing="ij")

    def smooth(n):
        f = np.zeros((B, n, H, W), np.float32)
        for b in range(B):
            for k in range(n):
                kx, ky, p = rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3), rng.uniform(0, 6.28)
                f[b, k] = rng.uniform(0.1, 0.6) * np.cos(kx * xx + ky * yy + p)
        return f

    x = np.empty((B, 5, H, W), np.float32)
    x[:, :3] = smooth(3) + 0.02 * rng.standard_normal((B, 3, H, W), np.float32)
    x[:, 3] = 0.6 + smooth(1)[:, 0]
    x[:, 4] = x[:, 3] > 0.15
    t = (2.0 * smooth(3) + 0.1 * rng.standard_normal((B, 3, H, W), np.float32)) * x[:, 4:5]
    return x, t.astype(np.float32)


class _Plane:
    """A device plane of a solver for torch (array interface).  A tensor made
    from it keeps it, and with it the solver that owns the memory."""

    def __init__(self, solver, ptr, shape, pitch, typestr, size):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": shape, "strides": (pitch * size, size), "typestr": typestr,
                                         "data": (ptr, False), "version": 2}


class _Views:
    """Views of a solver's resident arrays; an address is looked up on every
    call, since some arrays are double-buffered."""

    def __init__(self, solver):
        self.g, self.seen = solver, {}
        lib = solver.lib
        lib.fw_field_device.argtypes = [ct.c_void_p, ct.c_int, ct.POINTER(ct.c_void_p), ct.POINTER(ct.c_int)]
        self.ids = {n: lib.fw_field_id(n.encode()) for n in STATE}
        self.ptr, self.pitch = ct.c_void_p(), ct.c_int()

    def __call__(self):
        out = {}
        for n, i in self.ids.items():
            self.g._check(self.g.lib.fw_field_device(self.g.ctx, i, ct.byref(self.ptr), ct.byref(self.pitch)))
            key = (n, self.ptr.value)
            if key not in self.seen:
                whole = n in fwgpu.INTF
                size = 4 if whole else self.g.rb
                self.seen[key] = torch.as_tensor(_Plane(self.g, self.ptr.value, self.g.shape_of(n), self.pitch.value,
                                                        "<i4" if whole else "<f%d" % size, size), device="cuda")
            out[n] = self.seen[key]
        return out


class _Run:
    """What a program holds: solvers, their views, a batch, a network.  Each
    frees itself when nothing refers to it any more; a batch keeps its
    members, a view its solver."""

    def __init__(self, case, solvers=(), batch=None, net=None, x=None, t=None):
        self.case, self.solvers, self.batch, self.net, self.x, self.t = case, list(solvers), batch, net, x, t
        self.views = [_Views(g) for g in self.solvers]


def prepare(case, seed):
    torch.cuda.init()
    kind = case["kind"]
    if kind == "batch":
        gs = _members(case, seed)
        return _Run(case, gs, batch=fwgpu.Batch(gs))
    if kind in ("train", "predict"):
        x, t = _net_data(case, seed)
        params = fwcnn.init_params(seed, last_scale=1.0 if kind == "predict" else 0.1)
        return _Run(case, net=fwcnn.Net(case["N"], case["M"], case["B"], params), x=x, t=t)
    g = _solver(case, seed)
    net = None
    if kind == "learned":
        net = fwcnn.Net(case["N"], case["M"], 1, fwcnn.init_params(seed, last_scale=0.01))
        net.set_conserve(True)
    if kind == "output":
        g.step(2)
    return _Run(case, [g], net=net)


def _routine_step(g, c):
    """One step as the drop-in's main loop calls it."""
    g.save_stage0(1)
    g.exchange()
    clock = g.estimate_dt()
    g.save_stage0(2)
    for stage in (1, 2, 3):
        g.dispersion()
        g.fluxes()
        g.sources()
        g.estimate_huv(stage)
        g.update_mask()
        g.breaking()
        g.exchange()
        g.sponge()
    g.check_blowup()
    return clock


def run(state):
    c, kind = state.case, state.case["kind"]
    if kind == "train":
        loss, grad = state.net.train_step(state.x, state.t, 1e-4, want_grad=True)
        return {"loss": loss, "grad": grad}
    if kind == "predict":
        return state.net.forward(state.x)
    if kind == "batch":
        state.batch.step(c["steps"])
        return {str(k): {n: v for n, v in view().items() if n in ("Eta", "Ubar", "Vbar")}
                for k, view in enumerate(state.views)}
    g = state.solvers[0]
    if kind == "output":
        s = g.stats()
        return {"budget": s, "fields": {n: g.download(n) for n in OUTPUT}}
    if kind == "routines":
        dt, time = _routine_step(g, c)
    else:
        dt, time = g.step(c["steps"])
        if kind == "learned":
            state.net.correct(g)
    return {"dt": dt, "time": time, **state.views[0]()}


# ---- what a pass cannot do without ---------------------------------------------
def work(case):
    kind, m = case["kind"], case.get("M", 0) * case.get("N", 0)
    if kind in ("train", "predict"):
        cells = m * case["B"]
        if kind == "predict":  # five features in, three values out
            return {"bytes": cells * 4 * 8, "flops": cells * fwcnn.FLOP_PER_CELL}
        return {"bytes": cells * 4 * 8 + 4 * 5 * fwcnn.NPARAMS, "flops": 3 * cells * fwcnn.FLOP_PER_CELL}
    size = 8 if case["prec"] == "dp" else 4
    if kind == "output":  # surface, velocities, depth and mask read, four fields to the host
        return {"bytes": m * (5 * size + 4 * size), "flops": 12 * m}
    if kind == "batch":
        rows = np.random.default_rng(case["M"] * 1000 + case["N"])
        m = sum(int(rows.integers(case["M"] // 2, 3 * case["M"] // 2)) * int(
            rows.integers(case["N"] // 2, 3 * case["N"] // 2)) for _ in range(case["members"]))
    w = {"bytes": m * STEP_WORDS * size * case["steps"], "flops": m * STEP_FLOPS * case["steps"]}
    if kind == "learned":
        w["bytes"] += m * 4 * 14
        w["flops"] += m * fwcnn.FLOP_PER_CELL
    return w


# ---- values in 64 bits -----------------------------------------------------------
def _forward64(p, x):
    """The network of include/fwcnn.h, plain convolutions."""
    h = x
    for k in "1234":
        W, b = p["W" + k], p["b" + k]
        w = W.reshape(3, 3, W.shape[1], W.shape[2]).permute(3, 2, 0, 1)
        h = torch.nn.functional.conv2d(h, w, b, padding=1)
        if k != "4":
            h = torch.relu(h)
    return h


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "predict"):
        x, t = (torch.from_numpy(a).double() for a in _net_data(case, seed))
        flat = fwcnn.init_params(seed, last_scale=1.0 if kind == "predict" else 0.1)
        p = {k: torch.from_numpy(v.astype(np.float64)) for k, v in fwcnn.unflatten(flat).items()}
        if kind == "predict":
            return _forward64(p, x)
        for v in p.values():
            v.requires_grad_(True)
        loss = ((_forward64(p, x) - t) ** 2).mean()
        loss.backward()
        return {"loss": float(loss.detach()), "grad": torch.cat([p[k].grad.reshape(-1) for k, _ in fwcnn.SHAPES])}
    if kind != "output":
        return None
    # the budget of the state the run holds (two steps in), summed in 64 bits
    s = prepare(case, seed)
    g = s.solvers[0]
    f = {n: g.download(n)[3:-3, 3:-3].astype(np.float64) for n in OUTPUT + ("Depth",)}
    wet = f["MASK"] >= 1
    e, u, v, h = f["Eta"][wet], f["U"][wet], f["V"][wet], (f["Eta"] + f["Depth"])[wet]
    da = case["dx"] ** 2
    budget = {"mass_volume": e.sum() * da, "energy": (0.5 * h * (u * u + v * v) + 0.5 * 9.81 * e * e).sum() * da,
              "max_eta": e.max(), "min_eta": e.min(), "max_u": abs(u).max(), "max_v": abs(v).max(),
              "wet_cells": int(wet.sum())}
    return {"budget": {k: (float(b) if k != "wet_cells" else b) for k, b in budget.items()},
            "fields": {n: None for n in OUTPUT}}

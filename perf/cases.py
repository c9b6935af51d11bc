"""What is measured of this framework, and at which sizes.

Each case is one call sequence of a user's program through the package's
public entry points (osinco3d_amd.solver, .capi, .warmstart):

  steps     a short run of the device-resident solver from given fields:
            upload, then whole time steps (prediction, pressure solve,
            correction, diagnostics); forms fp64, mg and nn of bench.py on its
            Taylor-Green, mixing-layer and jet flows
  operators one step's operators of the drop-in on device arrays: the six
            derivatives of a component, predict_velocity, divergence,
            correct_velocity
  scalar    transeq, the passive scalar's transport step
  diagnose  the driver's output branch: statistics, rotational, Q criterion and
            function_stats on device arrays
  poisson   the multigrid pressure solver from zero (multigrid = 1)
  train     gradients of the warm-start network on one sample: forward, mean
            squared error, backward

`listed` holds the fixed cases, `draw` gives more of the same ranges,
`prepare` what a program has in hand, `run` one pass, `work` the bytes and
operations a pass cannot do without, `exact` the result in 64 bits from plain
torch.
"""
from __future__ import annotations

import ctypes
import math
import os

import numpy as np
import torch

from osinco3d_amd import capi, solver, warmstart
from osinco3d_amd.config import Config, jet_config, mixing_layer_config, tgv_config

WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(solver.__file__)), "warmstart_weights.npy")
TWO_PI = 2.0 * math.pi


def listed():
    return [
        # The smallest run: launches and latency only (the size of the smoke
        # test and of the quick parity runs).
        {"name": "steps_fp64_tgv16", "kind": "steps", "flow": "tgv", "form": "fp64", "nx": 16,
         "ny": 16, "nz": 16, "steps": 4, "scheme": 2},
        # The reference's own config 1: TGV 64^3, AB2, FP64.
        {"name": "steps_fp64_tgv64", "kind": "steps", "flow": "tgv", "form": "fp64", "nx": 64,
         "ny": 64, "nz": 64, "steps": 3, "scheme": 2},
        # The benchmark's TGV 256^3 in the drop-in's precision.
        {"name": "steps_fp64_tgv256", "kind": "steps", "flow": "tgv", "form": "fp64", "nx": 256,
         "ny": 256, "nz": 256, "steps": 1, "scheme": 3},
        # The benchmark's headline form: mixed precision, adaptive
        # extrapolation, coarse-grid correction, learned warm start.
        {"name": "steps_nn_tgv256", "kind": "steps", "flow": "tgv", "form": "nn", "nx": 256,
         "ny": 256, "nz": 256, "steps": 6, "scheme": 3},
        # The benchmark's mixing layer: LES, free-slip y, AB2.
        {"name": "steps_mg_mixing384", "kind": "steps", "flow": "mixing", "form": "mg", "nx": 384,
         "ny": 256, "nz": 128, "steps": 4, "scheme": 2},
        # The benchmark's planar jet, the largest run: x-Dirichlet ends, LES, AB3.
        {"name": "steps_mg_jet512", "kind": "steps", "flow": "jet", "form": "mg", "nx": 512,
         "ny": 384, "nz": 256, "steps": 3, "scheme": 3},
        # The drop-in's operators on the reference's published 185^3
        # free-slip TGV grid: odd sizes, partial tiles.
        {"name": "operators_185", "kind": "operators", "nx": 185, "ny": 185, "nz": 185, "wall": 3},
        # Scalar transport at the benchmark's size, walls in y.
        {"name": "scalar_256", "kind": "scalar", "nx": 256, "ny": 256, "nz": 256, "wall": 1},
        # The every-25-steps output branch of the driver at 256^3.
        {"name": "diagnose_256", "kind": "diagnose", "nx": 256, "ny": 256, "nz": 256, "wall": 0},
        # One pressure solve with multigrid = 1 (bench.py --workload poisson).
        {"name": "poisson_mg_256", "kind": "poisson", "nx": 256, "ny": 256, "nz": 256, "wall": 0},
        # One sample of train_warmstart's default training (128^3 runs, so a
        # 32^3 network) ...
        {"name": "train_32", "kind": "train", "nx": 32, "ny": 32, "nz": 32},
        # ... and of its jet training (512x384x256 over 4).
        {"name": "train_jet", "kind": "train", "nx": 128, "ny": 96, "nz": 64},
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(round(v / multiple)) * multiple)


def draw(rng):
    """A case of the listed ranges: log-uniform sizes per axis, odd ones where
    the entry point takes them."""
    kind = rng.choice(["steps", "steps", "steps", "operators", "scalar", "diagnose", "poisson",
                       "train"])
    if kind == "train":
        return {"kind": kind, "nx": _log_int(rng, 16, 128, 8), "ny": _log_int(rng, 16, 96, 8),
                "nz": _log_int(rng, 8, 64, 8)}
    if kind == "poisson":
        return {"kind": kind, "nx": _log_int(rng, 16, 384, 8), "ny": _log_int(rng, 16, 256, 2),
                "nz": _log_int(rng, 16, 256, 2), "wall": rng.choice([0, 1])}
    if kind != "steps":
        return {"kind": kind, "nx": _log_int(rng, 16, 384), "ny": _log_int(rng, 16, 256),
                "nz": _log_int(rng, 16, 256), "wall": rng.choice([0, 1, 3])}
    form = rng.choice(["fp64", "fp64", "mg", "mg", "nn"])
    flow = rng.choice(["tgv", "tgv", "mixing"]) if form == "fp64" else \
        rng.choice(["tgv", "mixing", "jet"])
    if form == "fp64":
        # The FP64 mixing layer sweeps to the stagnation rule: smaller grids.
        nx, ny, nz = (_log_int(rng, 16, 160 if flow == "tgv" else 96, 2) for _ in range(3))
        if flow == "tgv":
            ny = nz = nx
    elif form == "nn":
        nx, ny, nz = (_log_int(rng, 64, 256, 32) for _ in range(3))
        if flow == "tgv":
            ny = nz = nx
    else:
        nx, ny, nz = _log_int(rng, 32, 384, 8), _log_int(rng, 32, 256, 4), _log_int(rng, 32, 256, 4)
        if flow == "tgv":
            nx = ny = nz = _log_int(rng, 32, 256, 8)
    return {"kind": kind, "flow": flow, "form": form, "nx": nx, "ny": ny, "nz": nz,
            "steps": rng.choice([1, 2]) if form == "fp64" else rng.choice([3, 4, 5]),
            "scheme": rng.choice([2, 3])}


# ------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _rand(g, *shape):
    """Uniform in [-1, 1), float64, on the GPU."""
    return 2.0 * torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda") - 1.0


def _axis(n, length):
    return torch.arange(n, dtype=torch.float64, device="cuda") * (length / n)


def _periodic_fields(nx, ny, nz, g, amp=0.1):
    """Taylor-Green velocity and pressure on [0, 2 pi)^3 plus a few seeded
    shear waves of low wavenumber (divergence-free)."""
    x, y, z = _axis(nx, TWO_PI)[None, None, :], _axis(ny, TWO_PI)[None, :, None], \
        _axis(nz, TWO_PI)[:, None, None]
    c = _rand(g, 18).tolist()
    wave = lambda a, t, k, p: amp * a * torch.sin(k * t + math.pi * p)  # noqa: E731
    u = torch.sin(x) * torch.cos(y) * torch.cos(z) + wave(c[0], z, 2, c[1]) + wave(c[2], y, 3, c[3])
    v = -torch.cos(x) * torch.sin(y) * torch.cos(z) + wave(c[4], x, 2, c[5]) + \
        wave(c[6], z, 3, c[7])
    w = wave(c[8], x, 1, c[9]) + wave(c[10], y, 2, c[11]) + torch.zeros_like(u)
    p = (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0
    return [t.contiguous() for t in (u, v, w, p)]


def _wall_bc(wall):
    """0: periodic; 1: free-slip y; 3: free-slip on every axis."""
    return [int(wall == 3), int(wall >= 1), int(wall == 3)]


def _flow_config(case):
    nx, ny, nz, flow = case["nx"], case["ny"], case["nz"], case["flow"]
    if flow == "tgv":
        return tgv_config(nx, case["steps"], case["scheme"])
    if flow == "mixing":
        cfg = mixing_layer_config(nx, ny, nz, case["steps"],
                                  lengths=(60.0 * nx / 384, 40.0 * ny / 256, 20.0 * nz / 128))
    else:
        cfg = jet_config(nx, ny, nz, case["steps"])
    cfg.itscheme = case["scheme"]
    return cfg


def _flow_fields(case, cfg, g):
    """Initial u, v, w, p of a run, float64 on the GPU."""
    nx, ny, nz = cfg.nx, cfg.ny, cfg.nz
    shape = (nz, ny, nx)
    if case["flow"] == "tgv":
        return _periodic_fields(nx, ny, nz, g)
    y = cfg.y0 + torch.arange(ny, dtype=torch.float64, device="cuda") * cfg.spacing()[1]
    z = torch.zeros(shape, dtype=torch.float64, device="cuda")
    if case["flow"] == "mixing":
        # tanh profile and uniform noise of 5 %, as solver.mixing_layer.
        u = 0.5 * cfg.u0 * torch.tanh(2.0 * y / cfg.l0)[None, :, None]
        return [u + 0.05 * _rand(g, *shape), 0.05 * _rand(g, *shape), 0.05 * _rand(g, *shape), z]
    # The jet's profile and a seeded spanwise wave in its shear layers.
    prof = torch.from_numpy(solver.jet_profile(cfg, y.cpu().numpy())).cuda()
    c = _rand(g, 4).tolist()
    zz = torch.arange(nz, dtype=torch.float64, device="cuda") * (TWO_PI / nz)
    wave = 0.02 * (c[0] * torch.sin(zz + math.pi * c[1]) + c[2] * torch.sin(2 * zz +
                                                                           math.pi * c[3]))
    u = (prof[None, :, None] * (1.0 + wave)[:, None, None]).expand(shape).contiguous()
    return [u, z, z.clone(), z.clone()]


class _DeviceArray:
    """A solver field (Solver.field_ptr) as an array torch can take in place."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr,
                                         "data": (ptr, False), "version": 3}


def _field_view(s, which):
    """Solver field `which` as a torch tensor in place.  The tensor keeps the
    solver, whose end would free the field."""
    kind = "<f8" if which == 6 or s.precision == solver.FP64 else "<f4"
    t = torch.as_tensor(_DeviceArray(s.field_ptr(which), (s.cfg.nz, s.cfg.ny, s.cfg.nx), kind),
                        device="cuda")
    t.solver = s
    return t


def _prepare_steps(case, seed):
    g = _gen(seed)
    cfg = _flow_config(case)
    form = case["form"]
    if form == "fp64":
        s, net = solver.Solver(cfg, solver.FP64), None
    else:
        # The settings of bench.py's forms mg and nn.
        s = solver.Solver(cfg, solver.MIXED,
                          solver.WARM_LEARNED if form == "nn" else solver.WARM_EXTRAPOLATE,
                          coarse_cycles=2, smooth_sweeps=8, adaptive=1)
        net = None
        if form == "nn":
            net = warmstart.load_or_none(WEIGHTS, (cfg.nx, cfg.ny, cfg.nz))
            net.attach(s)
    fields = _flow_fields(case, cfg, g)
    if case["flow"] == "jet":
        s.set_inflow(*solver.jet_inflow(cfg, seed=int(seed) + 1))
    return {"solver": s, "net": net, "fields": fields, "views": {}}


def _run_steps(case, state):
    s = state["solver"]
    s.upload(*state["fields"])
    info = []
    for it in range(1, case["steps"] + 1):
        info.append(s.step(it))
    # p moves between the solver's pressure buffers: views by address.
    out = {}
    for which, name in ((0, "u"), (1, "v"), (2, "w"), (6, "p")):
        key = (which, s.field_ptr(which))
        if key not in state["views"]:
            state["views"][key] = _field_view(s, which)
        out[name] = state["views"][key]
    out["iterations"] = [i["sor_exit_iter"] for i in info]
    out["reasons"] = [i["sor_reason"] for i in info]
    # Extrema of the velocity, in its own precision.
    out["velocity"] = np.array([i["vel_min"] + i["vel_max"] + i["cfl"] for i in info],
                               np.float64 if s.precision == solver.FP64 else np.float32)
    return out


RE, DT, SC = 1600.0, 2e-3, 0.7
ADT = [DT, 3 * DT / 2, 23 * DT / 12]
BDT = [0.0, -DT / 2, -16 * DT / 12]
CDT = [0.0, 0.0, 5 * DT / 12]


def _spacing(case):
    bc = _wall_bc(case["wall"])
    n = (case["nx"], case["ny"], case["nz"])
    return tuple((math.pi / (m - 1)) if b else TWO_PI / m for m, b in zip(n, bc))


def _operator_fields(case, g):
    """Velocity, pressure of a TGV-like flow on the box of _spacing."""
    d = _spacing(case)
    t = [torch.arange(m, dtype=torch.float64, device="cuda") * h
         for m, h in zip((case["nx"], case["ny"], case["nz"]), d)]
    x, y, z = t[0][None, None, :], t[1][None, :, None], t[2][:, None, None]
    c = _rand(g, 8).tolist()
    u = torch.sin(x) * torch.cos(y) * torch.cos(z) + 0.1 * c[0] * torch.sin(2 * x) * \
        torch.cos(3 * z + 0 * y)
    v = -torch.cos(x) * torch.sin(y) * torch.cos(z) + 0.1 * c[1] * torch.sin(2 * y) * \
        torch.cos(2 * x + 0 * z)
    w = 0.2 * c[2] * torch.cos(x) * torch.cos(2 * y) * torch.sin(z)
    p = (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) * (1 + 0.1 * c[3]) / 16
    shape = u.shape
    # A little noise, as resolved small scales leave it.
    return [(f + 1e-3 * _rand(g, *shape)).contiguous() for f in (u, v, w, p)]


def _prepare_operators(case, seed):
    g = _gen(seed)
    u, v, w, p = _operator_fields(case, g)
    shape = tuple(u.shape)
    hist = [0.1 * _rand(g, 3, *shape) for _ in range(3)]
    new = lambda: torch.empty_like(u)  # noqa: E731
    return {"u": [u, v, w], "p": p, "hist": hist, "pred": [new() for _ in range(3)],
            "der": [new() for _ in range(6)], "div": new(), "out": [new() for _ in range(3)]}


def _der_codes(case):
    """First and second derivative of u along x, y, z: the routines schemes()
    binds for a component that is odd in x."""
    bc = _wall_bc(case["wall"])
    kind = [2 if bc[0] else 0, 1 if bc[1] else 0, 1 if bc[2] else 0]
    return [6 * a + 3 * o + kind[a] for a in range(3) for o in range(2)]


def _run_operators(case, s):
    d, bc = _spacing(case), _wall_bc(case["wall"])
    for q, which in enumerate(_der_codes(case)):
        capi.der(which, s["der"][q], s["u"][0], d[q // 2])
    capi.predict_velocity(s["pred"], s["u"], s["hist"], RE, ADT, BDT, CDT, 3, 3, d, 0, 0.17, 0.0,
                          None, bc)
    stats = capi.divergence(s["div"], *s["pred"], d, bc, odd=1, divisor=DT)
    _, vel = capi.correct_velocity(s["out"], s["pred"], s["p"], DT, d, bc)
    return {"der": s["der"], "pred": s["pred"], "hist": s["hist"], "div": s["div"],
            "stats": stats, "u": s["out"], "velocity": vel}


def _prepare_scalar(case, seed):
    g = _gen(seed)
    u, v, w, _ = _operator_fields(case, g)
    shape = tuple(u.shape)
    # A blob that spans the clipping bounds 0 and 1.
    phi = torch.clamp(0.5 + 0.7 * u * torch.sign(v) + 0.05 * _rand(g, *shape), 0.0, 1.0)
    return {"phi": phi, "u": [u, v, w], "src": 0.01 * _rand(g, *shape),
            "hist": 0.1 * _rand(g, 3, *shape)}


def _run_scalar(case, s):
    capi.transeq(s["phi"], s["u"], s["src"], s["hist"], RE, SC, ADT, BDT, CDT, 2, 2,
                 _spacing(case), 0, None, _wall_bc(case["wall"]))
    return {"phi": s["phi"], "hist": s["hist"]}


def _prepare_diagnose(case, seed):
    u, v, w, p = _operator_fields(case, _gen(seed))
    new = lambda: torch.empty_like(u)  # noqa: E731
    return {"u": [u, v, w], "p": p, "rot": [new() for _ in range(3)], "q": new()}


def _run_diagnose(case, s):
    d, bc = _spacing(case), _wall_bc(case["wall"])
    stats = capi.statistics(*s["u"], d, RE, 1.0, bc)
    # o3d_rotational and o3d_q_criterion on device arrays (the capi wrappers
    # allocate host arrays for their results).
    lib = capi.load()
    tail = [ctypes.c_double(h) for h in d] + [case["nx"], case["ny"], case["nz"],
                                              (ctypes.c_int * 3)(*bc)]
    vel = [capi.ptr(t) for t in s["u"]]
    capi.check(lib.o3d_rotational(*[capi.ptr(t) for t in s["rot"]], *vel, *tail))
    capi.check(lib.o3d_q_criterion(capi.ptr(s["q"]), *vel, *tail))
    return {"statistics": stats, "rot": s["rot"], "q": s["q"],
            "pressure": capi.function_stats(s["p"])}


def _prepare_poisson(case, seed):
    g = _gen(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    _, _, _, p = _operator_fields(case, g)
    # The divergence over dt of a predicted velocity: a smooth part and a rough one.
    rhs = 4.0 * (p - p.mean()) + 0.5 * _rand(g, *shape)
    return {"rhs": (rhs - rhs.mean()).contiguous(), "p": torch.empty_like(p)}


def _run_poisson(case, s):
    s["p"].zero_()
    cycles, rmax, reason = capi.poisson_multigrid(s["p"], s["rhs"], _spacing(case),
                                                  "0011" if case["wall"] else "0000", tol=1e-6,
                                                  max_cycles=100, with_reason=True)
    return {"p": s["p"], "cycles": cycles, "reason": reason}


def _prepare_train(case, seed):
    g = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    net = warmstart.Network(nx, ny, nz)
    net.load(WEIGHTS)
    # The two input planes (residual and previous increment, in units of the
    # increment's RMS) and the target: smooth fields with some roughness.
    u, v, w, p = _periodic_fields(nx, ny, nz, g, amp=0.5)
    incr = u + 0.3 * v * w + 0.05 * _rand(g, nz, ny, nx)
    incr = incr / incr.square().mean().sqrt()
    res = 0.2 * (p - p.mean()) + 0.1 * _rand(g, nz, ny, nx)
    tgt = incr + 0.25 * v + 0.3 * _rand(g, nz, ny, nx)
    flat = lambda t: t.reshape(-1).to(torch.float32).contiguous()  # noqa: E731
    inp = torch.stack([flat(res), flat(incr)])
    return {"net": net, "inp": inp, "tgt": flat(tgt), "out": torch.empty_like(inp[0]),
            "dout": torch.empty_like(inp[0]),
            "grads": torch.empty(net.nparam, dtype=torch.float32, device="cuda")}


def _run_train(case, s):
    net = s["net"]
    net.zero_grad()
    net.forward(s["inp"], s["out"])
    loss = net.mse(s["out"], s["tgt"], s["dout"])
    net.backward(s["dout"])
    capi.check(net.lib.o3d_nn_get_grads(net.h, capi.ptr(s["grads"])))
    return {"out": s["out"], "loss": loss, "grads": s["grads"]}


_PREPARE = {"steps": _prepare_steps, "operators": _prepare_operators, "scalar": _prepare_scalar,
            "diagnose": _prepare_diagnose, "poisson": _prepare_poisson, "train": _prepare_train}
_RUN = {"steps": _run_steps, "operators": _run_operators, "scalar": _run_scalar,
        "diagnose": _run_diagnose, "poisson": _run_poisson, "train": _run_train}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["case"] = dict(case)
    return state


def run(state):
    return _RUN[state["case"]["kind"]](state["case"], state)


# --------------------------------------------------------------------- work
def _net_flops(n):
    """Multiply-adds times two of the network's forward pass on n voxels."""
    spec = [(2, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2),
            (64, 128, 3), (128, 128, 3), (128, 64, 2), (64, 64, 2), (64, 32, 1), (32, 32, 1),
            (32, 16, 0), (16, 16, 0)]
    return sum(54.0 * ci * co * n / 8 ** lvl for ci, co, lvl in spec)


def work(case):
    n = float(case["nx"]) * case["ny"] * case["nz"]
    kind = case["kind"]
    if kind == "train":
        # Inputs, target, output, its gradient and the weight gradients;
        # forward, data gradient and weight gradient of every convolution.
        return {"bytes": 20.0 * n + 8.0 * 1320945, "flops": 3.0 * _net_flops(n)}
    if kind == "poisson":
        # rhs in, p out; a few full-grid sweeps and residuals per solve.
        return {"bytes": 16.0 * n, "flops": 5 * (9 * 10.0 + 20.0) * n}
    if kind == "diagnose":
        # Each of the four calls reads its inputs once; curl and Q are written.
        return {"bytes": 8.0 * n * (3 + 3 + 3 + 1 + 3 + 1), "flops": 360.0 * n}
    if kind == "scalar":
        # phi, u, src, one history slot in; phi and two history slots out.
        return {"bytes": 8.0 * n * (1 + 3 + 1 + 1 + 1 + 2), "flops": 70.0 * n}
    if kind == "operators":
        # Six derivatives (1 in, 1 out), predict (3 + 6 in, 3 + 9 out),
        # divergence (3 in, 1 out), correction (4 in, 3 out).
        return {"bytes": 8.0 * n * (12 + 9 + 12 + 4 + 7), "flops": 420.0 * n}
    es = 8.0 if case["form"] == "fp64" else 4.0
    k = case["steps"]
    # Per step: u in and out, the new and the old history terms, p in and
    # out; and the four uploaded fields once.
    per = es * (6 + 3 + 3 * (case["scheme"] - 1)) + 16.0
    return {"bytes": n * (k * per + 64.0),
            "flops": n * k * 320.0 + (k * _net_flops(n / 64) if case["form"] == "nn" else 0.0)}


# -------------------------------------------------------------------- exact
def _shift(f, axis, s, bc, odd):
    """f(. + s) along axis (0 x, 1 y, 2 z): periodic wrap, or the mirror about
    the end nodes, with a sign change of the mirrored values when odd."""
    dim = 2 - axis
    if not bc:
        return torch.roll(f, -s, dim)
    n = f.shape[dim]
    q = torch.arange(n, device=f.device) + s
    out = (q < 0) | (q > n - 1)
    q = torch.where(q < 0, -q, torch.where(q > n - 1, 2 * (n - 1) - q, q))
    r = f.index_select(dim, q)
    if odd:
        shape = [1, 1, 1]
        shape[dim] = n
        r = r * torch.where(out, -1.0, 1.0).to(f.dtype).reshape(shape)
    return r


def _d1(f, axis, h, bc, odd):
    t = [_shift(f, axis, s, bc, odd) for s in (1, 2, 3)]
    b = [_shift(f, axis, -s, bc, odd) for s in (1, 2, 3)]
    g = (45 * (t[0] - b[0]) - 9 * (t[1] - b[1]) + (t[2] - b[2])) / (60 * h)
    if bc and not odd:
        g.select(2 - axis, 0).zero_()
        g.select(2 - axis, f.shape[2 - axis] - 1).zero_()
    return g


def _d2(f, axis, h, bc, odd):
    near = _shift(f, axis, 1, bc, odd) + _shift(f, axis, -1, bc, odd)
    far = _shift(f, axis, 2, bc, odd) + _shift(f, axis, -2, bc, odd)
    return (16 * near - far - 30 * f) / (12 * h * h)


def _gradients(u, d, bc):
    return [[_d1(u[c], a, d[a], bc[a], c == a) for a in range(3)] for c in range(3)]


def _stats(f):
    nz, ny, nx = f.shape
    ix = int((f == f.max()).reshape(-1).nonzero()[0])
    return [float(f.min()), float(f.max()), float(f.mean()), ix % nx + 1, ix // nx % ny + 1,
            ix // (nx * ny) + 1]


def _tendency(u, d, bc, re, csd2):
    """F of the momentum equations, and its gradients."""
    g = _gradients(u, d, bc)
    nu = 1.0 / re
    if csd2:
        s2 = sum(g[a][a] ** 2 for a in range(3))
        s2 = s2 + 2 * sum((0.5 * (g[a][b] + g[b][a])) ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
        nu = nu + csd2 * torch.sqrt(2 * s2)
    return [nu * sum(_d2(u[c], a, d[a], bc[a], c == a) for a in range(3)) -
            sum(u[a] * g[c][a] for a in range(3)) for c in range(3)]


def _poisson(rhs, d, bc):
    """Solution of the 7-point problem (mirrored axes by even extension), up to
    a constant, by Fourier transforms."""
    n = rhs.shape
    w = torch.ones_like(rhs)
    for a in range(3):
        if bc[a]:
            for e in (0, n[2 - a] - 1):
                w.select(2 - a, e).mul_(0.5)
    f = rhs - (w * rhs).sum() / w.sum()
    for a in range(3):
        if bc[a]:
            dim = 2 - a
            f = torch.cat([f, f.flip(dim).narrow(dim, 1, n[dim] - 2)], dim)
    lam = 0
    for a in range(3):
        dim = 2 - a
        k = torch.arange(f.shape[dim], dtype=torch.float64, device=f.device)
        shape = [1, 1, 1]
        shape[dim] = f.shape[dim]
        lam = lam + ((2 * torch.cos(TWO_PI * k / f.shape[dim]) - 2) / d[a] ** 2).reshape(shape)
    lam[0, 0, 0] = 1.0
    F = torch.fft.fftn(f) / lam
    F[0, 0, 0] = 0
    return torch.fft.ifftn(F).real[: n[0], : n[1], : n[2]]


def _exact_steps(case, seed):
    if case["flow"] == "jet" or (case["flow"] == "mixing" and case["form"] == "fp64"):
        # The jet's inflow rules are the package's own; the FP64 mixing layer's
        # solve ends on the stagnation rule, off the solution.
        return None
    cfg = _flow_config(case)
    u = _flow_fields(case, cfg, _gen(seed))[:3]
    d, bc, dt = cfg.spacing(), cfg.bc(), cfg.time_step_overrides()
    csd2 = (cfg.cs * cfg.delta()) ** 2 if cfg.iles else 0.0
    ab = [[1.0], [1.5, -0.5], [23 / 12, -16 / 12, 5 / 12]]
    hist = []
    for it in range(1, case["steps"] + 1):
        hist = [_tendency(u, d, bc, cfg.re, csd2)] + hist[:2]
        co = ab[min(it, cfg.itscheme) - 1]
        up = [u[c] + dt * sum(k * h[c] for k, h in zip(co, hist)) for c in range(3)]
        rhs = sum(_d1(up[a], a, d[a], bc[a], True) for a in range(3)) / dt
        p = _poisson(rhs, d, bc)
        u = [up[a] - dt * _d1(p, a, d[a], bc[a], False) for a in range(3)]
    # The pressure is defined up to a constant; counts and extrema are not
    # computed values of their own.
    return {"u": u[0], "v": u[1], "w": u[2], "p": None, "iterations": None, "reasons": None,
            "velocity": None}


def _exact_operators(case, seed):
    s = _prepare_operators(case, seed)
    d, bc = _spacing(case), _wall_bc(case["wall"])
    u, hist = s["u"], s["hist"]
    der = []
    for a in range(3):
        der += [_d1(u[0], a, d[a], bc[a], a == 0), _d2(u[0], a, d[a], bc[a], a == 0)]
    F = _tendency(u, d, bc, RE, 0.0)
    # Slot 0 is replaced by this step's F, the older ones are read, then all
    # move down by one.
    pred = [u[c] + ADT[2] * F[c] + BDT[2] * hist[c][1] + CDT[2] * hist[c][2] for c in range(3)]
    new = [torch.stack([F[c], F[c], hist[c][1]]) for c in range(3)]
    div = sum(_d1(pred[a], a, d[a], bc[a], True) for a in range(3))
    out = [pred[a] - DT * _d1(s["p"], a, d[a], bc[a], False) for a in range(3)]
    vel = np.array([[float(f.min()), float(f.max()), float(f.abs().max()), 0.0] for f in out])
    return {"der": der, "pred": pred, "hist": new, "div": div / DT, "stats": None, "u": out,
            "velocity": vel}


def _exact_scalar(case, seed):
    s = _prepare_scalar(case, seed)
    d, bc = _spacing(case), _wall_bc(case["wall"])
    phi, u, hist = s["phi"], s["u"], s["hist"]
    F = sum(_d2(phi, a, d[a], bc[a], False) for a in range(3)) / (RE * SC) + s["src"] - \
        sum(u[a] * _d1(phi, a, d[a], bc[a], False) for a in range(3))
    new = phi + ADT[1] * F + BDT[1] * hist[1]
    c = new.clamp(0.0, 1.0)
    w = torch.minimum(c, 1.0 - c)
    c = (c + (new.mean() - c.mean()) * (w / w.sum())).clamp(0.0, 1.0)
    return {"phi": c, "hist": torch.stack([F, F, hist[2]])}


def _exact_diagnose(case, seed):
    s = _prepare_diagnose(case, seed)
    d, bc = _spacing(case), _wall_bc(case["wall"])
    u = s["u"]
    g = _gradients(u, d, bc)
    xnu = 1.0 / RE
    lap = [sum(_d2(u[c], a, d[a], bc[a], c == a) for a in range(3)) for c in range(3)]
    rot = [g[2][1] - g[1][2], g[0][2] - g[2][0], g[1][0] - g[0][1]]
    off = sum((g[a][b] + g[b][a]) ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
    mean = lambda t: float(t.mean())  # noqa: E731
    st = [1.0, mean(0.5 * sum(t * t for t in u)),
          mean(0.5 * xnu * (4 * sum(g[a][a] ** 2 for a in range(3)) + 2 * off)),
          mean(-xnu * sum(u[c] * lap[c] for c in range(3))),
          mean(0.5 * sum(r * r for r in rot))]
    st += [mean(t * t) for t in u] + [mean(g[c][a] ** 2) for c in range(3) for a in range(3)]
    q = -0.5 * sum(g[a][a] ** 2 for a in range(3)) - g[0][1] * g[1][0] - g[0][2] * g[2][0] - \
        g[1][2] * g[2][1]
    return {"statistics": np.array(st), "rot": rot, "q": q, "pressure": np.array(_stats(s["p"]))}


def _exact_train(case, seed):
    """The network in 64-bit sums with its activations, weights and
    activation gradients rounded to BF16 where its layers store them."""
    state = _prepare_train(case, seed)
    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    P = torch.from_numpy(state["net"].params()).cuda().double()
    bf = lambda t: t.to(torch.float32).to(torch.bfloat16).double()  # noqa: E731
    spec = [(16, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
            (128, 64), (64, 64), (64, 32), (32, 32), (32, 16), (16, 16)]
    offs, o = [], 0
    for ci, co in spec:
        offs.append((o, o + co * 27 * ci))
        o += co * 27 * ci + co
    taps = [(t, t % 3 - 1, t // 3 % 3 - 1, t // 9 - 1) for t in range(27)]
    G = torch.zeros_like(P)

    def weights(i):
        ci, co = spec[i]
        return bf(P[offs[i][0]:offs[i][1]]).reshape(co, 27, ci), P[offs[i][1]:offs[i][1] + co]

    def shifted(x, dx, dy, dz):
        return torch.roll(x, (-dz, -dy, -dx), (0, 1, 2))

    def layer(i, x, skip=None):
        W, b = weights(i)
        y = b.expand(x.shape[:3] + b.shape).clone()
        for t, dx, dy, dz in taps:
            y += (shifted(x, dx, dy, dz).reshape(-1, x.shape[3]) @
                  W[:, t, :].t().contiguous()).reshape(y.shape)
        if skip is not None:
            y = y + skip
        return bf(torch.where(y > 0, y, 0.1 * y))

    def pool(x):
        z, y, w, c = x.shape
        return bf(x.reshape(z // 2, 2, y // 2, 2, w // 2, 2, c).mean(dim=(1, 3, 5)))

    def up(x):
        return x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

    def up_t(g):
        z, y, w, c = g.shape
        return g.reshape(z // 2, 2, y // 2, 2, w // 2, 2, c).sum(dim=(1, 3, 5))

    def back(i, gy, y, x, want=True):
        """Gradients of layer i; returns (of its input, of its skip)."""
        ci, co = spec[i]
        d = gy * torch.where(y > 0, 1.0, 0.1)
        dz_ = bf(d)
        G[offs[i][1]:offs[i][1] + co] = d.sum(dim=(0, 1, 2))
        gw = G[offs[i][0]:offs[i][1]].reshape(co, 27, ci)
        W, _ = weights(i)
        flat = dz_.reshape(-1, co)
        gx = torch.zeros_like(x) if want else None
        for t, dx, dy, dz in taps:
            gw[:, t, :] = flat.t().contiguous() @ shifted(x, dx, dy, dz).reshape(-1, ci)
            if want:
                gx += (shifted(dz_, -dx, -dy, -dz).reshape(-1, co) @
                       W[:, t, :].contiguous()).reshape(gx.shape)
        return gx, d

    inp = state["inp"].double().reshape(2, nz, ny, nx)
    x = torch.zeros((nz, ny, nx, 16), dtype=torch.float64, device="cuda")
    x[..., 0], x[..., 1] = bf(inp[0]), bf(inp[1])
    e0a = layer(0, x)
    e0 = layer(1, e0a)
    p1 = pool(e0)
    e1a = layer(2, p1)
    e1 = layer(3, e1a)
    p2 = pool(e1)
    e2a = layer(4, p2)
    e2 = layer(5, e2a)
    p3 = pool(e2)
    e3a = layer(6, p3)
    e3 = layer(7, e3a)
    u2 = up(e3)
    d2a = layer(8, u2, e2)
    d2 = layer(9, d2a)
    u1 = up(d2)
    d1a = layer(10, u1, e1)
    d1 = layer(11, d1a)
    u0 = up(d1)
    d0a = layer(12, u0, e0)
    d0 = layer(13, d0a)
    head = P[o:o + 17]
    out = d0 @ head[:16] + head[16] + inp[1]
    diff = out - state["tgt"].double().reshape(nz, ny, nx)
    # The library forms the output and its gradient in 32 bits.
    dout = 2.0 * (out.float() - state["tgt"].reshape(nz, ny, nx)).double() / diff.numel()
    G[o:o + 16] = (dout[..., None] * d0).sum(dim=(0, 1, 2))
    G[o + 16] = dout.sum()
    g, _ = back(13, dout[..., None] * head[:16], d0, d0a)
    gu, g_e0 = back(12, g, d0a, u0)
    g, _ = back(11, up_t(gu), d1, d1a)
    gu, g_e1 = back(10, g, d1a, u1)
    g, _ = back(9, up_t(gu), d2, d2a)
    gu, g_e2 = back(8, g, d2a, u2)
    g, _ = back(7, up_t(gu), e3, e3a)
    g, _ = back(6, g, e3a, p3)
    g, _ = back(5, g_e2 + up(g) / 8, e2, e2a)
    g, _ = back(4, g, e2a, p2)
    g, _ = back(3, g_e1 + up(g) / 8, e1, e1a)
    g, _ = back(2, g, e1a, p1)
    g, _ = back(1, g_e0 + up(g) / 8, e0, e0a)
    back(0, g, e0a, x, want=False)
    # The first layer's padded input channels carry nothing.
    return {"out": out.reshape(-1), "loss": float(diff.square().mean()), "grads": G}


def exact(case, seed):
    # A multigrid solve ends on a residual bound, with the constant it
    # happens to reach: no value of its own in 64 bits.
    f = {"steps": _exact_steps, "operators": _exact_operators, "scalar": _exact_scalar,
         "diagnose": _exact_diagnose, "train": _exact_train}.get(case["kind"])
    return f(case, seed) if f else None

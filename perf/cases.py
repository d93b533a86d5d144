"""The work that a user of the column-physics engine has it do, as cases to
measure: which inputs, one pass through the public entry points, the bytes and
operations a pass cannot do without, and how close two answers have to be.

Two kinds of programs use the engine.  One holds a plan (``ColumnPhysics`` or
``ColumnEnsemble``), hands it host arrays, steps it and reads host arrays back;
a plan belongs to a grid, and the library keeps one at a time, so the plan is
kept here by the case and the states of one case differ in their tracers,
velocities and forcing.  The other holds device arrays and remaps them
(``roundabout_amd.rdb.remap``), or trains the closure network on host arrays
(``rdb_mlp_adam_steps``).
"""

from __future__ import annotations

import ctypes
import math
import os
import struct
import tempfile

import numpy as np
import torch

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnEnsemble, ColumnPhysics, _ffi, default_config
from roundabout_amd.rdb import remap as R

DT = 3600.0
LIVE = 1.5e-4  # a layer at most this thick is vanished
GRAV = 9.80665
WIDTHS = (381, 256, 256, 256, 256, 149)  # the closure network of 75 levels

# every contributor that is off at the defaults
CONTRIB = dict(epbl_enable=1, epbl_tke_diags=1, conv_enable=1, ddiff_enable=1, kv_ml_invz2=1.0e-2)
EPBL = dict(epbl_enable=1)


def listed():
    return [
        # the smallest program: a CPU-sized z-star basin, one day of hourly steps between two looks at it
        dict(name="day_small", kind="run", nx=64, ny=64, nz=20, topo="zstar", passive=2, steps=24, tune=False, split=False),
        # a host ocean model that calls the column physics once per thermodynamic step with its own arrays
        dict(name="coupled_step", kind="coupled", nx=160, ny=128, nz=75, topo="zlevel", passive=2, steps=1, tune=False, split=False),
        # an ocean tile on its own for ten days, tuned once
        dict(name="tile_10days", kind="run", nx=1440, ny=1080, nz=75, topo="zlevel", passive=2, steps=240, tune=True, split=False),
        # the energetic boundary layer in place of KPP, on a small basin
        dict(name="epbl_small", kind="contrib", nx=64, ny=64, nz=20, topo="zstar", passive=0, steps=24, knobs="epbl"),
        # every optional contributor on a regional grid, one day
        dict(name="contrib_regional", kind="contrib", nx=480, ny=360, nz=75, topo="zlevel", passive=2, steps=24, knobs="all"),
        # a one-dimensional ocean model: the column step and the vertical viscosity of the velocities, five days
        dict(name="momentum_regional", kind="momentum", nx=480, ny=360, nz=75, topo="zlevel", passive=0, steps=120, mom6=False),
        # an ensemble of small oceans of unlike size, ten days
        dict(name="ensemble_6", kind="ensemble", nx=160, ny=96, nz=50, members=6, passive=1, steps=240),
        # the learned closure with its guard, two days
        dict(name="surrogate_regional", kind="surrogate", nx=480, ny=360, nz=75, topo="zlevel", passive=2, steps=48),
        # training of the closure network on one batch
        dict(name="train_8192", kind="train", batch=8192, steps=100),
        # column remap of a small batch, as an embedding of the remap in another grid would call it
        dict(name="columns_small", kind="columns", ncol=1000, nz=33, method="ppm_h4", extrap=False, nonunif=False),
        # the ALE remap of an ocean tile after a step: four tracers (two with budget slots) and both face velocities
        dict(name="ale_tile", kind="ale", nx=1440, ny=1080, nz=75, topo="zlevel", method="ppm", passive=2, extrap=False,
             nonunif=False, ke=False, zfaces=False, check=False),
        # the high-order remap with every option, and its precondition checked first
        dict(name="ale_regional_pqm", kind="ale", nx=480, ny=360, nz=75, topo="zlevel", method="pqm", passive=0, extrap=True,
             nonunif=True, ke=True, zfaces=True, check=True),
    ]


def draw(rng):
    """One more case: any kind, sizes spread over the ranges between the listed ones, odd sizes as likely as even."""
    kind = rng.choice(["run", "run", "coupled", "contrib", "momentum", "ensemble", "surrogate", "train", "columns", "ale", "ale"])
    topo = rng.choice(["zstar", "zlevel"])
    nz = rng.randint(8, 90)

    def grid(most):
        n = _log(rng, 64 * 64, most)
        nx = max(9, round(math.sqrt(n) * rng.uniform(0.7, 1.6)))
        return dict(nx=nx, ny=max(7, n // nx), nz=nz, topo=topo)

    if kind == "train":
        return dict(kind=kind, batch=_log(rng, 512, 8192), steps=rng.randint(20, 100))
    if kind == "columns":
        return dict(kind=kind, ncol=_log(rng, 100, 200000), nz=nz, method=rng.choice(sorted(R.METHODS)),
                    extrap=rng.random() < 0.5, nonunif=rng.random() < 0.5)
    if kind == "ale":
        return dict(kind=kind, **grid(400000), method=rng.choice(sorted(R.METHODS)), passive=rng.randint(0, 3),
                    extrap=rng.random() < 0.5, nonunif=rng.random() < 0.5, ke=rng.random() < 0.5, zfaces=rng.random() < 0.5,
                    check=rng.random() < 0.5)
    if kind == "ensemble":
        return dict(kind=kind, nx=_log(rng, 40, 200), ny=_log(rng, 40, 150), nz=nz, members=rng.randint(2, 8),
                    passive=rng.randint(0, 3), steps=rng.randint(24, 240))
    if kind == "surrogate":
        return dict(kind=kind, **grid(200000), passive=rng.randint(0, 3), steps=rng.randint(12, 48))
    if kind == "momentum":
        return dict(kind=kind, **grid(200000), passive=0, steps=rng.randint(24, 120), mom6=rng.random() < 0.5)
    if kind == "contrib":
        return dict(kind=kind, **grid(170000), passive=rng.randint(0, 5), steps=rng.randint(6, 24), knobs=rng.choice(["epbl", "all"]))
    if kind == "coupled":
        return dict(kind=kind, **grid(60000), passive=rng.randint(0, 3), steps=1, tune=False, split=rng.random() < 0.3)
    return dict(kind=kind, **grid(300000), passive=rng.randint(0, 5), steps=rng.randint(24, 240), tune=rng.random() < 0.3,
                split=rng.random() < 0.3)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# --------------------------------------------------------------- grids
_GRIDS: dict = {}
_PLAN: dict = {"key": None, "plan": None}


def _members(case):
    """The grids of a case: one, or an ensemble's members of unlike size."""
    if case["kind"] != "ensemble":
        return [(case["nx"], case["ny"], case["nz"], case["topo"])]
    return [(max(8, case["nx"] * (4 + m % 3) // 5), max(8, case["ny"] * (5 - m % 2) // 5), max(4, case["nz"] * (3 + m % 3) // 5),
             "zlevel" if m % 2 else "zstar") for m in range(case["members"])]


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps")))


def _grid(nx, ny, nz, topo, passive=0):
    """Geometry of one grid (the same for every seed): an Ocean without its tracers, and the layer centres' depth on the GPU."""
    key = (nx, ny, nz, topo)
    if key not in _GRIDS:
        for k in [k for k in _GRIDS if _GRIDS[k][0].h.size > 2e7]:
            del _GRIDS[k]
        if topo == "zstar":
            o = synth.make_ocean(nx, ny, nz, 11, land_frac=0.1, topo=topo, n_passive=0)
        else:
            o = synth.make_ocean(nx, ny, nz, 11, land_frac=0.3, topo=topo, dmin=50.0, dmax=5500.0, n_passive=0)
        o.T = o.S = None
        _GRIDS[key] = (o, _dev(o.wet))
    return _GRIDS[key]


def _dev(a):
    """A Fortran-ordered host array as a C-ordered (levels, ny, nx) tensor on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()


def _host(t):
    """Such a tensor as a Fortran-ordered host array."""
    return t.cpu().numpy().T


def _state(case, o, wet, seed, passive):
    """Tracers and forcing of one grid, drawn on the GPU as synth draws them; smooth and stably stratified below the surface
    for the learned closure, whose guard hands unstable columns to the plain path."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + o.nx * 31 + o.nz)

    def normal(*s):
        return torch.randn(*s, generator=g, device="cuda", dtype=torch.float64)

    def uniform(*s):
        return torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)

    h = _dev(o.h)
    nz, ny, nx = h.shape
    z = torch.flip(torch.cumsum(torch.flip(h, (0,)), 0), (0,)) - 0.5 * h
    amp = 10.0 + 18.0 * uniform(ny, nx)
    T = 2.0 + amp * torch.exp(-z / 500.0)
    if case["kind"] == "surrogate":
        T = T - 4.0e-4 * z + 0.002 * normal(nz, ny, nx)
        S = 34.5 + 0.5 * (1.0 - torch.exp(-z / 700.0)) + 0.002 * normal(nz, ny, nx)
    else:
        T = T + 0.1 * normal(nz, ny, nx)
        S = 35.0 + 0.3 * normal(nz, ny, nx)
    w = wet > 0.5
    f = {"temperature": T * w, "salinity": S * w}
    for i in range(passive):
        f["tracer_%d" % (i + 1)] = uniform(nz, ny, nx) * w
    f = {k: _host(v) for k, v in f.items()}
    ax, ay = 6.283185307179586 * uniform(ny, nx + 1), 6.283185307179586 * uniform(ny + 1, nx)
    f["tau_x"] = _host(0.08 * torch.exp(0.5 * normal(ny, nx + 1)) * torch.cos(ax))
    f["tau_y"] = _host(0.08 * torch.exp(0.5 * normal(ny + 1, nx)) * torch.sin(ay))
    f["Q_heat"] = _host(-50.0 + 100.0 * normal(ny, nx))
    f["Q_salt"] = np.zeros((nx, ny), order="F")
    f["bl_depth"] = np.zeros((nx, ny), order="F")
    if case["kind"] in ("coupled", "momentum"):
        scale = 0.8 + 0.4 * float(uniform(1))
        f["u_face_x_layer"], f["v_face_y_layer"] = np.asfortranarray(o.u * scale), np.asfortranarray(o.v * scale)
    if case["kind"] == "coupled":
        f["h_layer"] = np.asfortranarray(np.where(o.h > LIVE, o.h * (0.99 + 0.02 * float(uniform(1))), o.h))
    return f


# --------------------------------------------------------------- plans
def _network(case):
    """A closure network for the grid's levels, written the way mlp_save writes one and loaded as a user loads his: random
    weights, outputs around the diffusivities and boundary-layer depths that the plain path gives."""
    nz = case["nz"]
    widths = (5 * nz + 6, 256, 256, 256, 256, 2 * nz - 1)
    rng = np.random.default_rng(4)
    parts = []
    for a, b in zip(widths[:-1], widths[1:]):
        parts += [rng.standard_normal(a * b) * math.sqrt(1.5 / a), 0.05 * rng.standard_normal(b)]
    level = np.ones(nz)
    fmean = np.concatenate([-2.0 * level, 0.0 * level, 0.0 * level, 0.0 * level, 1.2 * level, [0.08, -50.0, 0.0, 8e-5, 0.01, 2800.0]])
    fstd = np.concatenate([2.0 * level, 0.5 * level, 1.5 * level, 1.5 * level, 2.5 * level, [0.05, 100.0, 1.0, 3e-5, 0.01, 1600.0]])
    far = np.full(widths[0], 1.0e30)
    nf = nz - 1
    stats = [fmean, fstd, -far, far, np.concatenate([np.full(nf, -4.0), np.full(nf, -3.3), [45.0]]),
             np.concatenate([np.full(nf, 0.5), np.full(nf, 0.4), [20.0]]),
             np.concatenate([np.full(nf, -5.0), np.full(nf, -4.0), [5.0]]), np.concatenate([np.full(nf, -1.0), np.full(nf, -1.0), [200.0]])]
    fd, path = tempfile.mkstemp(suffix=".rdbsurr")
    with os.fdopen(fd, "wb") as f:
        f.write(b"RDBSURR5" + struct.pack("<4i", nz, widths[0], widths[-1], len(widths)) + struct.pack("<6i", *widths))
        for p in parts + stats:
            f.write(np.asarray(p, dtype=np.float32).tobytes())
    return path


def _plan(case):
    """The plan of a case's grid, made when another one was in hand."""
    key = _key(case)
    if _PLAN["key"] == key:
        return _PLAN["plan"]
    if _PLAN["plan"] is not None:
        _PLAN["plan"].close()
    _PLAN.update(key=None, plan=None)
    cfg = default_config()
    for k, v in {"epbl": EPBL, "all": CONTRIB}.get(case.get("knobs"), {}).items():
        setattr(cfg, k, v)
    if case.get("split"):
        cfg.precision = _ffi.PREC_SPLIT
    grids = [_grid(*m)[0] for m in _members(case)]
    if case["kind"] == "ensemble":
        plan = ColumnEnsemble([(o.nx, o.ny, o.nz, o.wet) for o in grids], n_passive=case["passive"], config=cfg,
                              sort_keys=[o.n_live for o in grids])
        for m, o in enumerate(grids):
            for name, a in (("h_layer", o.h), ("u_face_x_layer", o.u), ("v_face_y_layer", o.v)):
                plan.member_set_field(m, name, a)
    else:
        o = grids[0]
        plan = ColumnPhysics(o.nx, o.ny, o.nz, o.wet, n_passive=case["passive"], config=cfg, k_top=o.k_top, sort_key=o.n_live)
        for name, a in (("h_layer", o.h), ("u_face_x_layer", o.u), ("v_face_y_layer", o.v), ("coriolis", o.coriolis)):
            plan.set_field(name, a)
    if case["kind"] == "surrogate":
        path = _network(case)
        plan.mlp_load(path)
        os.unlink(path)
        plan.set_guard(_ffi.GUARD_SURFACE)
        plan.set_closure(_ffi.CLOSURE_SURROGATE)
    if case.get("tune"):
        plan.autotune(DT)
    _PLAN.update(key=key, plan=plan)
    return plan


# ------------------------------------------------------- device arrays
class _Shared:
    """A DeviceArray as torch sees it."""

    def __init__(self, d):
        self.keep = d
        self.__cuda_array_interface__ = {"shape": d.shape[::-1], "typestr": "<f8", "data": (d.ptr.value, False), "version": 2}


def _device(t):
    """(DeviceArray, its tensor) with the values of a (levels, ..) tensor."""
    d = R.DeviceArray(tuple(t.shape)[::-1])
    v = torch.as_tensor(_Shared(d), device="cuda")
    v.copy_(t)
    return d, v


def _ale_pair(h, seed):
    """(h_old, h_new) after a step of layered dynamics, as synth.ale_pair: jittered layers under a free-surface anomaly, and
    the z-star target of the same column total."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 104729 + 3)
    nz, ny, nx = h.shape
    live = h > LIVE
    H, HL = h.sum(0), (h * live).sum(0)
    a = 1.2 + float(torch.rand(1, generator=g, device="cuda"))
    eta = a * torch.sin(torch.linspace(0.0, 3.0, nx, device="cuda", dtype=torch.float64))[None, :] \
        * torch.cos(torch.linspace(0.0, 2.0, ny, device="cuda", dtype=torch.float64))[:, None]
    eta = eta * (HL > 0)
    ho = h * (1.0 + 0.05 * (torch.rand(nz, ny, nx, generator=g, device="cuda", dtype=torch.float64) - 0.5))
    ho = torch.where(live, ho, h)
    ho = torch.where(live, ho * ((HL + eta) / (ho * live).sum(0).clamp_min(1e-300)), h)
    hn = torch.where(live, h * ((H + eta) / H.clamp_min(1e-300)), h)
    top = torch.where(live, torch.arange(nz, device="cuda")[:, None, None], -1).amax(0).clamp_min(0)
    hn.scatter_add_(0, top[None], (ho.sum(0) - hn.sum(0))[None])
    return ho, hn


# ------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        rng = np.random.default_rng(seed)
        B = case["batch"]
        parts = []
        for a, b in zip(WIDTHS[:-1], WIDTHS[1:]):
            parts += [rng.standard_normal(a * b, dtype=np.float32) * np.float32(math.sqrt(2.0 / a)), np.zeros(b, np.float32)]
        x = rng.standard_normal((B, WIDTHS[0]), dtype=np.float32)
        t = np.tanh(x[:, :WIDTHS[-1]] + 0.5 * x[:, -WIDTHS[-1]:])
        w = (rng.random((B, WIDTHS[-1])) < 0.75).astype(np.float32)  # a quarter of a column's interfaces lie below its bed
        return {"case": case, "params": np.concatenate(parts), "x": x, "t": np.ascontiguousarray(t), "w": w}
    if kind == "columns":
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed))
        nz, n = case["nz"], case["ncol"]

        def rand(*s):
            return torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)

        ho = 1.0 + 99.0 * rand(nz, n)
        hn = ho * (0.9 + 0.2 * rand(nz, n))
        hn = hn * (ho.sum(0) / hn.sum(0))
        q = torch.cumsum(rand(nz, n), 0) + 0.3 * rand(nz, n)
        s = {"case": case}
        for name, t in (("ho", ho), ("hn", hn), ("q", q), ("out", torch.zeros_like(q))):
            s[name], s[name + "_t"] = _device(t)
        torch.cuda.synchronize()
        return s
    if kind == "ale":
        o, wet = _grid(case["nx"], case["ny"], case["nz"], case["topo"])
        h = _dev(o.h)
        ho, hn = _ale_pair(h, seed)
        s = {"case": case, "tracers": [], "budgets": []}
        s["ho"], s["ho_t"] = _device(ho)
        s["hn"], s["hn_t"] = _device(hn)
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed) * 13 + 1)
        w = wet > 0.5
        z = torch.flip(torch.cumsum(torch.flip(h, (0,)), 0), (0,)) - 0.5 * h
        for i in range(2 + case["passive"]):
            r = torch.randn(h.shape, generator=g, device="cuda", dtype=torch.float64)
            s["tracers"].append(_device(((2.0 + 18.0 * torch.exp(-z / 500.0) + 0.1 * r) if i == 0 else (35.0 + 0.3 * r)) * w))
            s["budgets"].append(_device(torch.zeros_like(h)) if i < 2 else None)
        for name, a in (("u", o.u), ("v", o.v)):
            f = _dev(a)
            s[name], s[name + "_t"] = _device(f + 0.02 * (f != 0) * torch.randn(f.shape, generator=g, device="cuda", dtype=torch.float64))
        torch.cuda.synchronize()
        return s
    _plan(case)
    members = []
    for i, m in enumerate(_members(case)):
        members.append(_state(case, *_grid(*m), seed * 17 + i, case["passive"]))
    torch.cuda.synchronize()
    return {"case": case, "fields": members}


# ----------------------------------------------------------------- run
def _tracers(case):
    return ["temperature", "salinity"] + ["tracer_%d" % (i + 1) for i in range(case["passive"])]


def _results(case):
    """What a program reads back: the tracers and the boundary layer, and what its kind of program needs besides."""
    kind = case["kind"]
    if kind == "contrib":
        return _tracers(case) + ["kv", "kt", "ks", "mld"]
    if kind == "momentum":
        return _tracers(case) + ["u_face_x_layer", "v_face_y_layer", "bl_depth"]
    if kind == "coupled":
        return _tracers(case) + ["kv", "kt", "ks", "bl_depth"]
    return _tracers(case) + ["bl_depth"] + (["kt"] if case["nx"] < 1000 else [])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        return _run_train(state)
    if kind == "columns":
        R.remap_column(state["ho"], state["hn"], state["q"], case["method"], bnd_extrap=case["extrap"], nonunif=case["nonunif"],
                       q_new=state["out"])
        return state["out_t"]
    if kind == "ale":
        return _run_ale(state)
    plan = _plan(case)
    if kind == "ensemble":
        for m, f in enumerate(state["fields"]):
            for name, a in f.items():
                plan.member_set_field(m, name, a)
        plan.step(DT, case["steps"])
        return [{n: plan.member_get_field(m, n) for n in _results(case)} for m in range(plan.n_members)]
    for name, a in state["fields"][0].items():
        plan.set_field(name, a)
    if kind == "momentum":
        for _ in range(case["steps"]):
            plan.step(DT, 1)
            plan.vdiff_momentum(DT, implicit_stress=1, hvel_mom6=int(case["mom6"]))
    else:
        plan.step(DT, case["steps"])
    return {n: plan.get_field(n) for n in _results(case)}


def _run_ale(s):
    c = s["case"]
    out = []
    if c["check"]:
        out += list(R.ocean_remap_scan_preconditions(s["ho"], s["hn"]))
    opt = dict(bnd_extrap=c["extrap"], nonunif=c["nonunif"])
    for (d, t), b in zip(s["tracers"], s["budgets"]):
        R.ocean_remap_tracer_field(s["ho"], s["hn"], d, c["method"], budget=b and b[0], **opt)
        out.append(t)
        if b:
            out.append(b[1])
    R.ocean_apply_ale_remap_faces(s["ho"], s["hn"], s["u"], s["v"], c["method"], conserve_ke=c["ke"], zlevel_faces=c["zfaces"], **opt)
    return out + [s["u_t"], s["v_t"]]


def _run_train(s):
    fp = ctypes.POINTER(ctypes.c_float)
    out = np.empty_like(s["params"])
    w = (ctypes.c_int * len(WIDTHS))(*WIDTHS)
    p = [s[k].ctypes.data_as(fp) for k in ("params", "x", "t", "w")]
    lib = _ffi.load()
    _ffi.check(lib.rdb_mlp_adam_steps(w, len(WIDTHS), p[0], s["case"]["batch"], p[1], p[2], p[3], s["case"]["steps"], 1e-3, 0.9, 0.999,
                                      1e-8, out.ctypes.data_as(fp)), lib)
    return out


# ---------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind == "train":
        n = sum(a * b for a, b in zip(WIDTHS[:-1], WIDTHS[1:]))
        per = case["batch"] * (2 * WIDTHS[0] + 8 * WIDTHS[-1]) + 28 * n
        return {"bytes": per * case["steps"], "flops": 6 * n * case["batch"] * case["steps"]}
    if kind == "columns":
        return {"bytes": 32 * case["ncol"] * case["nz"], "flops": 60 * case["ncol"] * case["nz"]}
    if kind == "ale":
        cells = case["nx"] * case["ny"] * case["nz"]
        nf = 2 + case["passive"]
        return {"bytes": 8 * cells * (2 * nf + 2 * 2 + 4 + 2), "flops": 60 * cells * (nf + 2)}
    total = {"bytes": 0.0, "flops": 0.0}
    for m in _members(case):
        o, _ = _grid(*m)
        live, wet, n = float(o.n_live.sum()), float(o.n_wet), case["passive"]
        step = 8.0 * ((8 + 2 * n) * live + (live + wet) * 3) + 44 * wet + (8.0 * 8 * o.h.size if kind == "momentum" else 0.0)
        flops = live * (180 + 12 * n)
        if kind == "surrogate":
            k = (5 * case["nz"] + 6) * 256 + 3 * 256 * 256 + 256 * (2 * case["nz"] - 1)
            step, flops = step + 8.0 * 2 * live, flops + 2.0 * k * wet
        host = 8.0 * o.h.size * (2 * (2 + n) + {"coupled": 6, "momentum": 4, "contrib": 3}.get(kind, 1))
        total["bytes"] += step * case["steps"] + host
        total["flops"] += flops * case["steps"]
    return total


# ----------------------------------------------------------- tolerance
def tolerance(case):
    # FP64 with the reference's operations in the reference's order: every correct implementation gives the same bits.  The
    # same holds of the single-precision assembly.
    if case["kind"] == "train":
        # bf16 operands, 32-bit sums, after up to 100 Adam steps
        return {"rel": 1.0e-2, "max": 0.9}
    if case["kind"] == "surrogate":
        # bf16 activations: a last bit in one of them moves log10 kt by 1e-3 and more; the tracers hardly move
        return {"rel": 1.0e-2, "max": 0.9}
    return "exact"


# --------------------------------------------------------------- exact
def exact(case, seed):
    """The same outputs from plain torch in 64 bits; None where the scheme is one that has no short plain form (EPBL and its
    companions, the fourth-order and quartic remaps, a network whose bf16 rounding feeds back into the state), and for runs
    too long for it."""
    kind = case["kind"]
    if kind == "train":
        return _exact_train(prepare(case, seed))
    if kind in ("columns", "ale"):
        if case["method"] not in ("pcm", "plm", "ppm"):
            return None
        return _exact_columns(case, seed) if kind == "columns" else _exact_ale(case, seed)
    if kind in ("run", "coupled", "ensemble", "momentum"):
        if case.get("split") or case.get("mom6") or case["steps"] * sum(m[2] for m in _members(case)) > 4000:
            return None
        o = [_grid(*m) for m in _members(case)]
        f = [_state(case, g, w, seed * 17 + i, case["passive"]) for i, (g, w) in enumerate(o)]
        got = [_exact_run(case, g, x) for (g, _), x in zip(o, f)]
        return got if kind == "ensemble" else got[0]
    return None


def _rho(T, S, h):
    a0 = 7.057924e-4 + 3.480336e-7 * T - 1.112733e-7 * S
    p0 = 5.790749e8 + 3.516535e6 * T - 4.002714e4 * T**2 + 2.084372e2 * T**3 + 5.944068e5 * S - 9.643486e3 * S * T
    la = 1.704853e5 + 7.904722e2 * T - 7.984422 * T**2 + 5.140652e-2 * T**3 - 2.302158e2 * S - 3.079464 * S * T
    return torch.where(h > LIVE, p0 / (la + a0 * p0), torch.full_like(h, 1035.0))


def _thomas(a, b, c, r):
    """Tridiagonal solve over the levels; r: a list of right-hand sides."""
    nz = b.shape[0]
    cp, x = torch.empty_like(b), [torch.empty_like(b) for _ in r]
    for k in range(nz):
        piv = b[k] - a[k] * cp[k - 1] if k else b[k]
        cp[k] = c[k] / piv
        for i, y in enumerate(r):
            x[i][k] = (y[k] - a[k] * x[i][k - 1]) / piv if k else y[k] / piv
    for k in range(nz - 2, -1, -1):
        for y in x:
            y[k] -= cp[k] * y[k + 1]
    return x


def _exact_run(case, o, f):
    rho0, cp_w, HV = 1035.0, 3992.0, LIVE
    h = _dev(f.get("h_layer", o.h))
    u, v = _dev(f.get("u_face_x_layer", o.u)), _dev(f.get("v_face_y_layer", o.v))
    wet, qh = _dev(o.wet), _dev(f["Q_heat"])
    tx, ty = _dev(f["tau_x"]), _dev(f["tau_y"])
    tr = [_dev(f[n]) for n in _tracers(case)]
    bl = _dev(f["bl_depth"])
    nz = h.shape[0]
    live = h > HV
    k_of = torch.arange(nz, device="cuda")[:, None, None]
    ksfc = torch.where(live.any(0), torch.where(live, k_of, -1).amax(0), nz - 1)
    at = lambda x: x.gather(0, ksfc[None])[0]  # noqa: E731
    tau = torch.sqrt((0.5 * (tx[:, :-1] + tx[:, 1:]))**2 + (0.5 * (ty[:-1] + ty[1:]))**2)
    hc = h.clamp_min(HV)
    kv = kt = None
    for _ in range(case["steps"]):
        uc, vc = 0.5 * (u[:, :, :-1] + u[:, :, 1:]), 0.5 * (v[:, :-1] + v[:, 1:])
        rho = _rho(tr[0], tr[1], h)
        dz = 0.5 * (h[:-1] + h[1:])
        sh2 = (((uc[1:] - uc[:-1]) / dz)**2 + ((vc[1:] - vc[:-1]) / dz)**2).clamp_min(1e-10)
        den = 1.0 + 5.0 * (-(GRAV * (rho[1:] - rho[:-1]) / (rho0 * dz)) / sh2).clamp_min(0.0)
        kv, kt = torch.zeros(nz + 1, *h.shape[1:], device="cuda", dtype=torch.float64), None
        kt = kv.clone()
        kv[1:nz], kt[1:nz] = 1e-4 + 1e-2 / den**2, 1e-5 + 1e-2 / den**3
        # KPP: bulk Richardson crossing from the first live layer down
        us, qT = torch.sqrt(tau / rho0), qh / (rho0 * cp_w)
        B0 = GRAV / rho0 * 1.7e-4 * qT
        ws = torch.sqrt(us**2 + ((-B0).clamp_min(0.0) * bl).pow(1.0 / 3.0)**2)
        u_r, v_r, b_r, d_r = at(uc), at(vc), -(GRAV * at(rho) / rho0), 0.5 * at(h)
        hb = (h * (k_of <= ksfc)).sum(0)
        done, ri_p, d_p, d, h_up = torch.zeros_like(wet, dtype=torch.bool), torch.zeros_like(wet), d_r, d_r, at(h)
        for k in range(nz - 2, -1, -1):
            on = (k < ksfc) & ~done
            dk = torch.where(on, d + 0.5 * (h_up + h[k]), d)
            db, dd = b_r + GRAV * rho[k] / rho0, torch.where(on, dk - d_r, torch.ones_like(d))
            vt2 = 6.0 * dk * torch.sqrt((db / dd).clamp_min(0.0)) * ws
            ri = db * dd / ((uc[k] - u_r)**2 + (vc[k] - v_r)**2 + vt2).clamp_min(1e-10)
            hit = on & (ri >= 0.3)
            fr = torch.where((ri - ri_p).abs() > 1e-12, (0.3 - ri_p) / torch.where(hit, ri - ri_p, torch.ones_like(ri)), torch.full_like(ri, 0.5))
            hb = torch.where(hit, d_p + fr * (dk - d_p), hb)
            done |= hit
            d, h_up = dk, torch.where(k < ksfc, h[k], h_up)
            ri_p, d_p = torch.where(on, ri, ri_p), torch.where(on, dk, d_p)
        bl = hb
        ws = torch.sqrt(us**2 + ((-B0).clamp_min(0.0) * hb).pow(1.0 / 3.0)**2)
        depth = torch.flip(torch.cumsum(torch.flip(h * (k_of <= ksfc), (0,)), 0), (0,))
        sg = depth[1:] / hb.clamp_min(1e-300)
        inside = (k_of[1:] <= ksfc) & (depth[1:] < hb) & (hb > 0) & (ws > 0)
        G = torch.where(inside, sg * (1.0 - sg)**2, torch.zeros_like(sg))
        kv[1:nz], kt[1:nz] = torch.maximum(kv[1:nz], hb * ws * G), torch.maximum(kt[1:nz], hb * ws * G)
        gam = 6.3 * G * qT * (B0 < 0)
        kv[1:nz], kt[1:nz] = kv[1:nz].clamp_min(1e-4), kt[1:nz].clamp_min(1e-5)
        # surface deposit, implicit diffusion, non-local transport
        src = torch.where(at(h) > HV, DT / (rho0 * cp_w) * qh * wet / at(h), torch.zeros_like(wet))
        tr[0] = tr[0].scatter_add(0, ksfc[None], src[None])
        face = DT * kt[1:nz] / (0.5 * (hc[:-1] + hc[1:])) * (live[:-1] & live[1:])
        lo, up = torch.zeros_like(h), torch.zeros_like(h)
        lo[1:], up[:-1] = face / hc[1:], face / hc[:-1]
        tr = _thomas(-lo, 1.0 + up + lo, -up, tr)
        fl = torch.zeros_like(kv)
        fl[1:nz] = gam * (live[:-1] & live[1:])
        tr[0] = torch.where(live, tr[0] + DT * (fl[1:] - fl[:-1]) / h, tr[0])
        if case["kind"] == "momentum":
            u, v = _viscosity(u, h, kv, tx, wet, 2), _viscosity(v, h, kv, ty, wet, 1)
    got = dict(zip(_tracers(case), tr), kv=kv, kt=kt, ks=kt, bl_depth=bl, u_face_x_layer=u, v_face_y_layer=v)
    return {n: _host(got[n]) for n in _results(case)}


def _viscosity(u, h, kv, tau, wet, dim):
    """Vertical viscosity of the faces along dim, arithmetic face thickness, wind stress in the top row."""
    def faces(x):
        d = dim - 3
        n = x.shape[d]
        return torch.cat([x.narrow(d, 0, 1), x], d), torch.cat([x, x.narrow(d, n - 1, 1)], d)
    a, b = faces(h)
    hf = (0.5 * (a + b)).clamp_min(LIVE)
    a, b = faces(kv)
    nz = h.shape[0]
    face = DT * (0.5 * (a + b))[1:nz] / (0.5 * (hf[:-1] + hf[1:]))
    lo, up = torch.zeros_like(hf), torch.zeros_like(hf)
    lo[1:], up[:-1] = face / hf[1:], face / hf[:-1]
    a, b = faces(wet[None])
    r = u.clone()
    r[-1] += DT * tau * torch.minimum(a, b)[0] / 1035.0 / hf[-1].clamp_min(1e-3)
    return _thomas(-lo, 1.0 + up + lo, -up, [r])[0]


def _half_jump(h_self, h_nbr, dq):
    d = dq * h_self / (h_self + h_nbr).clamp_min(1e-30)
    return torch.copysign(torch.minimum(d.abs(), dq.abs()), d)


def _reconstruct(case, h, q):
    """Cell parabolas (left, right, curvature) of the piecewise methods: q(x) = L + x (R - L + q6 (1 - x))."""
    nz, be, m = h.shape[0], case["extrap"], case["method"]
    zero = torch.zeros_like(q)
    if nz == 1 or m == "pcm":
        return q, q, zero
    E = 1.0e-20

    def jump():
        hl, hc, hr = h[:-2], h[1:-1], h[2:]
        return hc / (hl + hc + hr + E) * ((2 * hl + hc) / (hc + hr + E) * (q[2:] - q[1:-1]) + (hc + 2 * hr) / (hl + hc + E) * (q[1:-1] - q[:-2]))

    end0, end1 = _half_jump(h[0], h[1], q[1] - q[0]), _half_jump(h[-1], h[-2], q[-1] - q[-2])
    if m == "plm" or nz == 2:
        s = zero.clone()
        dl, dr = q[1:-1] - q[:-2], q[2:] - q[1:-1]
        if case["nonunif"]:
            sc = jump()
            lo, hi = torch.minimum(torch.minimum(q[:-2], q[2:]), q[1:-1]), torch.maximum(torch.maximum(q[:-2], q[2:]), q[1:-1])
            w = 0.5 * torch.copysign(torch.minimum(sc.abs(), 2 * torch.minimum(q[1:-1] - lo, hi - q[1:-1])), sc)
        else:
            w = 0.5 * torch.copysign(torch.minimum(dl.abs(), dr.abs()), dl)
        s[1:-1] = torch.where(dl * dr > 0, w, zero[1:-1])
        if be:
            s[0], s[-1] = end0, end1
        return q - s, q + s, zero
    e = torch.empty(nz + 1, *q.shape[1:], device=q.device, dtype=q.dtype)  # edge values
    e[0], e[nz] = q[0], q[-1]
    if case["nonunif"]:
        for k in (1, nz - 1):
            e[k] = (q[k - 1] * h[k] + q[k] * h[k - 1]) / (h[k - 1] + h[k] + E)
        j = jump()
        h0, h1, h2, h3 = h[:-3], h[1:-2], h[2:-1], h[3:]
        dq, i12 = q[2:-1] - q[1:-2], 1.0 / (h1 + h2 + E)
        wa, wb = (h0 + h1) / (2 * h1 + h2 + E), (h2 + h3) / (h1 + 2 * h2 + E)
        e[2:nz - 1] = q[1:-2] + h1 * i12 * dq + (2 * h1 * h2 * i12 * (wa - wb) * dq - h1 * wa * j[1:] + h2 * wb * j[:-1]) / (h0 + h1 + h2 + h3 + E)
    else:
        e[1], e[nz - 1] = 0.5 * (q[0] + q[1]), 0.5 * (q[-2] + q[-1])
        e[2:nz - 1] = 7.0 / 12.0 * (q[1:-2] + q[2:-1]) - 1.0 / 12.0 * (q[:-3] + q[3:])
    qm, qp = torch.cat([q[:1], q[:-1]]), torch.cat([q[1:], q[-1:]])
    lo, hi = torch.minimum(torch.minimum(qm, qp), q), torch.maximum(torch.maximum(qm, qp), q)
    L, Rt = torch.maximum(lo, torch.minimum(hi, e[:-1])), torch.maximum(lo, torch.minimum(hi, e[1:]))
    flat, dq, t6 = (q - L) * (Rt - q) <= 0, Rt - L, 6 * q - 3 * (L + Rt)
    steep = ~flat & (t6.abs() > dq.abs())
    L2 = torch.where(steep & (t6 * dq > 0), 3 * q - 2 * Rt, L)
    R2 = torch.where(steep & ~(t6 * dq > 0), 3 * q - 2 * L, Rt)
    L, Rt = torch.where(flat, q, L2), torch.where(flat, q, R2)
    q6 = 6 * q - 3 * (L + Rt)
    if be:
        for k, d in ((0, end0), (nz - 1, end1)):
            L[k], Rt[k], q6[k] = q[k] - d, q[k] + d, 0.0
    return L, Rt, q6


def _overlaps(ho, hn):
    """Pairs (target, source, bottom, top, source bottom) whose overlap is positive somewhere."""
    zo = torch.cat([torch.zeros_like(ho[:1]), torch.cumsum(ho, 0)])
    zn = torch.cat([torch.zeros_like(hn[:1]), torch.cumsum(hn, 0)])
    for k in range(hn.shape[0]):
        for j in range(ho.shape[0]):
            lo, hi = torch.maximum(zn[k], zo[j]), torch.minimum(zn[k + 1], zo[j + 1])
            if bool((hi > lo).any()):
                yield k, j, lo, hi, zo[j]


def _integral(L, Rt, q6, q, h, j, lo, hi, z0):
    hs = h[j].clamp_min(1e-300)
    a, b = (lo - z0) / hs, (hi - z0) / hs
    v = h[j] * ((b - a) * L[j] + 0.5 * (b * b - a * a) * (Rt[j] - L[j] + q6[j]) - (b**3 - a**3) * q6[j] / 3.0)
    return torch.where(hi > lo, v, torch.zeros_like(v))


def _remap(case, ho, hn, q):
    P = _reconstruct(case, ho, q)
    out = torch.zeros_like(q)
    for k, j, lo, hi, z0 in _overlaps(ho, hn):
        out[k] += _integral(*P, q, ho, j, lo, hi, z0)
    return torch.where(hn > 0, out / hn, torch.zeros_like(out))


def _exact_columns(case, seed):
    s = prepare(case, seed)
    return _remap(case, s["ho_t"], s["hn_t"], s["q_t"])


def _donor(h, c):
    """The column with each vanished layer holding its nearest live neighbour's value, from above first."""
    out, nz = torch.zeros_like(c), h.shape[0]
    have = torch.zeros_like(h[0], dtype=torch.bool)
    cur = torch.zeros_like(c[0])
    for k in range(nz - 1, -1, -1):
        on = h[k] > LIVE
        cur, have = torch.where(on, c[k], cur), have | on
        out[k] = cur
    top = torch.zeros_like(c[0])
    for k in range(nz):
        top = torch.where(h[k] > LIVE, c[k], top)
    seen = torch.zeros_like(have)
    for k in range(nz - 1, -1, -1):
        seen |= h[k] > LIVE
        out[k] = torch.where(seen, out[k], torch.where(have, top, torch.zeros_like(top)))
    return out


def _exact_ale(case, seed):
    s = prepare(case, seed)
    ho, hn = s["ho_t"], s["hn_t"]
    nz, out = ho.shape[0], []
    if ho.numel() > 4.0e7 or nz < 2:
        return None
    if case["check"]:
        a, b = ho.sum(0), hn.sum(0)
        rel = float(((b - a).abs() / torch.maximum(a.abs(), b.abs()).clamp_min(1e-20)).max())
        out += [0, None if rel < 1e-12 else rel, 0.0]
    for (_, c), bud in zip(s["tracers"], s["budgets"]):
        d = _donor(ho, c)
        P = _reconstruct(case, ho, d)
        dm, dp = torch.cat([d[:1], d[:-1]]), torch.cat([d[1:], d[-1:]])
        lo_s, hi_s = torch.minimum(torch.minimum(dm, dp), d), torch.maximum(torch.maximum(dm, dp), d)
        if case["extrap"]:
            for k, n in ((0, 1), (nz - 1, nz - 2)):
                lo_s[k], hi_s[k] = torch.minimum(lo_s[k], 2 * d[k] - d[n]), torch.maximum(hi_s[k], 2 * d[k] - d[n])
        ex = torch.where(ho <= LIVE, c - d, torch.zeros_like(c))
        lo_s, hi_s = lo_s + ex, hi_s + ex
        q, lo_t, hi_t = torch.zeros_like(c), torch.full_like(c, math.inf), torch.full_like(c, -math.inf)
        for k, j, lo, hi, z0 in _overlaps(ho, hn):
            on = hi > lo
            q[k] += _integral(*P, d, ho, j, lo, hi, z0) + torch.where(on, ex[j] * (hi - lo), torch.zeros_like(lo))
            lo_t[k] = torch.where(on, torch.minimum(lo_t[k], lo_s[j]), lo_t[k])
            hi_t[k] = torch.where(on, torch.maximum(hi_t[k], hi_s[j]), hi_t[k])
        q = torch.maximum(lo_t, torch.minimum(hi_t, q / hn))
        out.append(q)
        if bud:
            out.append(hn * q - ho * c)
    for name, dim in (("u_t", 2), ("v_t", 1)):
        w = s[name]
        pair = []
        for x in (ho, hn):
            n = x.shape[dim]
            a, b = torch.cat([x.narrow(dim, 0, 1), x], dim), torch.cat([x, x.narrow(dim, n - 1, 1)], dim)
            pair.append(torch.minimum(a, b) if case["zfaces"] else 0.5 * (a + b))
        if case["zfaces"]:
            gone = (pair[0] <= LIVE) | (pair[1] <= LIVE)
            pair = [p.masked_fill(gone, 0.0) for p in pair]
        fo, fn = pair
        un = _remap(case, fo, fn, w)
        if case["ke"]:
            so, sn = fo.sum(0), fn.sum(0)
            uo, ub = (fo * w).sum(0) / so.clamp_min(1e-300), (fn * un).sum(0) / sn.clamp_min(1e-300)
            ko, kn = (0.5 * fo * (w - uo)**2).sum(0), (0.5 * fn * (un - ub)**2).sum(0)
            ok = (so > LIVE) & (sn > LIVE) & (ko > 0) & (kn > 0)
            un = torch.where(ok, ub + torch.sqrt(ko / kn.clamp_min(1e-300)).clamp_max(1.25) * (un - ub), un)
        out.append(un)
    return out


def _exact_train(s):
    """The same Adam steps on float64 weights and activations."""
    p, at, layers = torch.from_numpy(s["params"]).double().cuda(), 0, []
    for a, b in zip(WIDTHS[:-1], WIDTHS[1:]):
        layers.append((p[at:at + a * b].view(b, a).clone().requires_grad_(), p[at + a * b:at + a * b + b].clone().requires_grad_()))
        at += a * b + b
    flat = [x for wb in layers for x in wb]
    x, t, w = (torch.from_numpy(s[k]).double().cuda() for k in ("x", "t", "w"))
    m, v = [torch.zeros_like(q) for q in flat], [torch.zeros_like(q) for q in flat]
    for n in range(1, s["case"]["steps"] + 1):
        y = x
        for i, (wt, b) in enumerate(layers):
            y = y @ wt.t() + b
            if i + 1 < len(layers):
                y = torch.nn.functional.gelu(y, approximate="tanh")
        g = torch.autograd.grad((w * (y - t)**2).sum() / w.sum(), flat)
        with torch.no_grad():
            for q, a, c, d in zip(flat, m, v, g):
                a.mul_(0.9).add_(0.1 * d)
                c.mul_(0.999).add_(0.001 * d * d)
                q -= 1e-3 * (a / (1 - 0.9**n)) / (torch.sqrt(c / (1 - 0.999**n)) + 1e-8)
    return torch.cat([q.detach().reshape(-1) for q in flat]).cpu().numpy()

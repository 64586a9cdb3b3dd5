"""The work a user of this framework has it do, as cases that can be timed and compared.

``listed()`` gives the standing cases, ``draw(rng)`` one more of the same
ranges, ``prepare(case, seed)`` what a program holds before the call (fields on
the GPU and the solver handle), ``run(state)`` one pass through the public
entry points, ``work(case)`` the bytes and operations the path cannot do
without, and ``exact(case, seed)`` the same outputs in 64 bits from dense
operators and torch's transforms, without this package's code.

Fields are torch tensors of shape (nz, ny, nx), which is the library's Fortran
order with x fastest.
"""
import ctypes as C
import math

import numpy as np
import torch

from chapsim2_amd import _lib
from chapsim2_amd.domain import (FFT_2DECOMP_3DFFT, FFT_FISHPACK_2DFFT, IACCU_CD2, IACCU_CD4, IACCU_CP4, IACCU_CP6,
                                 IBC_DIRICHLET, IBC_PERIODIC, PREC_FP64, PREC_MIXED, PROJ_EXACT, PROJ_REFERENCE,
                                 Batch, Domain)
from chapsim2_amd.initial import HEATED_H_RANGE, heated_channel_table
from chapsim2_amd.mlp import NP as MLP_NP
from chapsim2_amd.mlp import Surrogate
from chapsim2_amd.props import PROPS_MLP, PROPS_TABLE, PropertyTable

LX, LZ = 4.0 * math.pi, 4.0 * math.pi / 3.0  # the channel's domain, y in [-1, 1]
DT = 5e-4
SMOOTH = sorted(2 ** a * 3 ** b * 5 ** c for a in range(10) for b in range(6) for c in range(4)
                if 8 <= 2 ** a * 3 ** b * 5 ** c <= 512)


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # Taylor-Green vortex, triply periodic 64^3: the reference's own test
        # flow; ten steps between two looks at the fields
        {"name": "tgv_fp64", "kind": "tgv", "nx": 64, "ny": 64, "nz": 64, "steps": 10},
        # a channel as small as a set-up check or a regression test runs it, stepped
        # as the reference's loop does: after each step the mass-conservation windows
        # and the velocity range are read back.  Launches and latency are all there is
        {"name": "channel_small", "kind": "loop", "nx": 32, "ny": 24, "nz": 16, "acc": IACCU_CD2, "steps": 5},
        # the plane channel at Re_tau 180, FP64, projection exact to round-off
        {"name": "channel_fp64", "kind": "channel", "nx": 256, "ny": 128, "nz": 256, "mixed": False,
         "beta": 1.5, "steps": 2},
        # the same in the mixed form, the flagship workload
        {"name": "channel_mixed", "kind": "channel", "nx": 256, "ny": 128, "nz": 256, "mixed": True,
         "beta": 1.5, "steps": 2},
        # a parameter study: uneven channels advanced together as one graph
        {"name": "batch_mixed", "kind": "batch", "count": 6, "grids": 7, "steps": 3},
        # the variable-property channel (energy equation, property table, variable
        # density and viscosity)
        {"name": "heated_mixed", "kind": "heated", "nx": 192, "ny": 96, "nz": 160, "steps": 1},
        # the compact operators called one by one, as a program that brings its own
        # time integration or post-processing does; FP64 at the channel's size
        {"name": "operators_fp64", "kind": "ops", "nx": 256, "ny": 128, "nz": 256, "f32": False, "acc": IACCU_CP6},
        # and FP32 on the large grid
        {"name": "operators_fp32", "kind": "ops", "nx": 512, "ny": 256, "nz": 512, "f32": True, "acc": IACCU_CP6},
        # the pressure solve (FFT in x and z, tridiagonal along y) on the large grid
        {"name": "poisson_fp64", "kind": "poisson", "nx": 512, "ny": 256, "nz": 512, "f32": False},
        # thermal properties of every cell from rho*h by the table
        {"name": "properties_table", "kind": "props", "cells": 256 * 128 * 256, "surrogate": False},
        # and by the neural surrogate attached to the table
        {"name": "properties_surrogate", "kind": "props", "cells": 128 * 72 * 144, "surrogate": True},
        # training the surrogate: forward, backward and Adam steps
        {"name": "surrogate_train", "kind": "train", "batch": 4096, "steps": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, lo, hi, even=False):
    """A transform length (2, 3, 5-smooth; even: twice one) spread over the logarithm of [lo, hi]."""
    want = _log(rng, lo, hi)
    every = [2 * v for v in SMOOTH if lo <= 2 * v <= hi] if even else [v for v in SMOOTH if lo <= v <= hi]
    return min(every, key=lambda v: (abs(v - want), v))


def draw(rng):
    kind = rng.choice(["tgv", "loop", "channel", "channel", "batch", "heated", "ops", "ops", "poisson", "poisson",
                       "props", "train"])
    if kind == "tgv":
        return {"kind": kind, "nx": _near(rng, 16, 128, True), "ny": _near(rng, 16, 128), "nz": _near(rng, 16, 128),
                "steps": rng.randint(1, 10)}
    if kind == "loop":
        return {"kind": kind, "nx": _near(rng, 16, 96, True), "ny": rng.randint(12, 64), "nz": _near(rng, 12, 64),
                "acc": rng.choice([IACCU_CD2, IACCU_CD2, IACCU_CP6]), "steps": 1 + rng.randint(0, 1)}
    if kind == "channel":
        return {"kind": kind, "nx": _near(rng, 24, 256, True), "ny": _log(rng, 24, 144), "nz": _near(rng, 16, 256),
                "mixed": rng.random() < 0.5, "beta": round(rng.uniform(1.0, 2.0), 3), "steps": rng.randint(1, 2)}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(2, 6), "grids": rng.randint(100, 10 ** 6), "steps": rng.randint(1, 3)}
    if kind == "heated":
        return {"kind": kind, "nx": _near(rng, 24, 192, True), "ny": _log(rng, 24, 96), "nz": _near(rng, 16, 160),
                "steps": 1}
    if kind in ("ops", "poisson"):
        c = {"kind": kind, "nx": _near(rng, 24, 512, True), "ny": _log(rng, 24, 256), "nz": _near(rng, 16, 512),
             "f32": rng.random() < 0.5}
        return dict(c, acc=rng.choice([IACCU_CP6, IACCU_CP6, IACCU_CP4, IACCU_CD4])) if kind == "ops" else c
    if kind == "props":
        sur = rng.random() < 0.4
        return {"kind": kind, "cells": _log(rng, 1000, 1_300_000 if sur else 8_000_000), "surrogate": sur}
    return {"kind": "train", "batch": _log(rng, 256, 8192), "steps": rng.randint(1, 3)}


def _grids(case):
    """The batch's uneven grids: sizes between 64 and 192 x 128 x 192, stretching and bulk Reynolds number of their own."""
    import random

    r = random.Random(case["grids"])
    return [{"nc": (r.choice([64, 72, 80, 96, 100, 128, 144, 160, 192]), r.choice(range(64, 129, 8)),
                    r.choice([64, 72, 80, 96, 100, 128, 144, 160, 192])),
             "beta": round(r.uniform(1.0, 2.0), 3), "ren": r.choice([2800.0, 6900.0])} for _ in range(case["count"])]


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _rand(seed, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1)


def _mesh_y(ny, beta):
    """yp, yc and dy/ds-inverses at nodes and centres of the two-sided tanh mesh on [-1, 1]."""
    def at(eta):
        y = np.tanh(beta * (eta - 0.5)) / math.tanh(0.5 * beta)
        return y, math.tanh(0.5 * beta) / beta / (1.0 - (y * math.tanh(0.5 * beta)) ** 2)

    yp, mp = at(np.arange(ny + 1) / ny)
    yc, mc = at((np.arange(ny) + 0.5) / ny)
    return yp, yc, mp, mc


def _channel_fields(nc, beta, seed):
    """Laminar profile, 10 % noise, unit bulk velocity; wall-normal velocity zero at the walls; a smooth pressure."""
    nx, ny, nz = nc
    yc, mc = (torch.from_numpy(v).cuda() for v in _mesh_y(ny, beta)[1::2])
    qx = 0.1 * _rand(4 * seed, nz, ny, nx) + 1.5 * (1.0 - yc * yc)[None, :, None]
    w = (1.0 / mc) / (1.0 / mc).sum()
    qx /= (qx.mean(dim=(0, 2)) * w).sum()
    qy = 0.1 * _rand(4 * seed + 1, nz, ny + 1, nx)
    qy[:, 0] = 0.0
    qy[:, -1] = 0.0
    qz = 0.1 * _rand(4 * seed + 2, nz, ny, nx)
    x = (torch.arange(nx, device="cuda", dtype=torch.float64) + 0.5) * (2 * math.pi / nx)
    z = (torch.arange(nz, device="cuda", dtype=torch.float64) + 0.5) * (2 * math.pi / nz)
    pr = 0.05 * torch.cos(2 * x)[None, None, :] * torch.cos(z)[:, None, None] * (1 - yc * yc)[None, :, None]
    return [t.contiguous() for t in (qx, qy, qz, pr)]


def _tgv_fields(nc, seed):
    """The Taylor-Green vortex with a small seeded disturbance (a divergence remains for the projection to remove)."""
    x, y, z = ((torch.arange(n, device="cuda", dtype=torch.float64)) * (2 * math.pi / n) for n in nc)
    xc, yc, zc = (t + math.pi / n for t, n in zip((x, y, z), nc))

    def prod(fz, fy, fx):
        return fz[:, None, None] * fy[None, :, None] * fx[None, None, :]

    qx = prod(zc.cos(), yc.cos(), x.sin())
    qy = -prod(zc.cos(), y.sin(), xc.cos())
    qz = torch.zeros_like(qx)
    pr = (torch.cos(2 * xc)[None, None, :] + torch.cos(2 * yc)[None, :, None]) * (torch.cos(2 * zc)[:, None, None] + 2) / 16
    q = [t + 0.01 * _rand(4 * seed + i, *qx.shape) for i, t in enumerate((qx, qy, qz))]
    return [t.contiguous() for t in q + [pr]]


def _channel_cfg(beta, **kw):
    return dict(dict(lxx=LX, lyb=-1.0, lyt=1.0, lzz=LZ, istret=2, rstret=beta / 20.0, dt=DT, ren=2800.0, idriven=1), **kw)


def _table_columns(pt):
    return {k: torch.from_numpy(np.ascontiguousarray(pt[:, c])).cuda() for k, c in
            (("h", 1), ("t", 2), ("d", 3), ("m", 4), ("k", 5), ("cp", 6))}


def _interp(x, xs, ys):
    """Linear interpolation on rising xs."""
    i = (torch.searchsorted(xs, x.contiguous(), right=True) - 1).clamp_(0, xs.numel() - 2)
    w = (xs[i + 1] - x) / (xs[i + 1] - xs[i])
    return w * ys[i] + (1 - w) * ys[i + 1]


def _rhoh(h, col):
    return _interp(h, col["h"], col["d"] * col["h"])


def _surrogate_params(tab, norm, seed):
    """Weights of a fitted 1-64-64-5 network: random tanh layers, the output layer by least squares on the table."""
    r = np.random.RandomState(seed % (1 << 31))
    w1, b1 = r.uniform(-3.0, 3.0, 64), r.uniform(-2.0, 2.0, 64)
    w2, b2 = r.uniform(-0.4, 0.4, (64, 64)), r.uniform(-0.2, 0.2, 64)
    x = (tab[:, 1] - norm[0]) / norm[1]
    a = np.tanh(np.tanh(np.outer(x, w1) + b1) @ w2.T + b2)
    y = (tab[:, [2, 3, 4, 5, 6]] - norm[2:7]) / norm[7:12]
    a1 = np.concatenate([a, np.ones((len(x), 1))], axis=1)
    w3 = np.linalg.solve(a1.T @ a1 + 1e-4 * len(x) * np.eye(65), a1.T @ y)
    p = np.concatenate([w1, b1, w2.ravel(), b2, w3[:64].T.ravel(), w3[64]]).astype(np.float32)
    assert p.size == MLP_NP
    return p


# --------------------------------------------------------------------------
# prepare and run
# --------------------------------------------------------------------------
def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _set(dm, fields):
    _lib.check(dm.lib.chs_set_state(dm.h, *[_ptr(t) for t in fields], _lib.MEM_DEVICE))


def _get(dm, fields):
    _lib.check(dm.lib.chs_get_state(dm.h, *[_ptr(t) for t in fields], _lib.MEM_DEVICE))


def _operators(case):
    """(direction, kind, input shape, output shape, walls' values given) of the operators a staggered solver applies."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cell = {0: (nx, ny, nz), 1: (nx, ny, nz), 2: (nx, ny, nz)}
    node = {0: (nx, ny, nz), 1: (nx, ny + 1, nz), 2: (nx, ny, nz)}
    return [(d, k, (cell if k in (0, 4) else node)[d], (node if k in (0, 4) else cell)[d], d == 1 and k in (0, 4))
            for d in range(3) for k in (0, 4, 1, 5)]  # C2P: interpolation, derivative; P2C: the same


def _op_inputs(case, seed):
    """A cell field, a node field along y and the wall values (nx, 4, nz) of the former, smooth with some noise."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dt = torch.float32 if case["f32"] else torch.float64

    def field(n2, k):
        x, y, z = (torch.arange(n, device="cuda", dtype=torch.float64) * (2 * math.pi / n) for n in (nx, n2, nz))
        f = torch.sin(3 * x + k)[None, None, :] * torch.cos(y)[None, :, None] * torch.cos(2 * z - k)[:, None, None]
        return (f + 0.05 * _rand(3 * seed + k, nz, n2, nx)).to(dt)

    c = field(ny, 0)
    wall = torch.stack([c[:, 0], c[:, -1], c[:, 0], c[:, -1]], dim=1) * 0.5
    return c, field(ny + 1, 1), wall.contiguous()


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind in ("tgv", "loop", "channel", "heated", "ops", "poisson"):
        nc = (case["nx"], case["ny"], case["nz"])
    if kind == "tgv":
        p2 = 2 * math.pi
        s["dm"] = Domain(nc, p2, 0.0, p2, p2, periodic_y=True, dt=1e-3, ren=1600.0, poisson=FFT_2DECOMP_3DFFT)
        s["in"] = _tgv_fields(nc, seed)
    elif kind == "loop":
        s["dm"] = Domain(nc, **_channel_cfg(1.5, iacc=case["acc"], projection=_loop_projection(case)))
        s["in"] = _channel_fields(nc, 1.5, seed)
    elif kind == "channel":
        s["dm"] = Domain(nc, **_channel_cfg(case["beta"], projection=PROJ_EXACT,
                                            precision=PREC_MIXED if case["mixed"] else PREC_FP64))
        s["in"] = _channel_fields(nc, case["beta"], seed)
    elif kind == "batch":
        grids = _grids(case)
        s["batch"] = Batch([_channel_cfg(g["beta"], nc=g["nc"], ren=g["ren"], projection=PROJ_EXACT,
                                         precision=PREC_MIXED) for g in grids])
        s["in"] = [_channel_fields(g["nc"], g["beta"], 100 * seed + i) for i, g in enumerate(grids)]
        for dm, f in zip(s["batch"].domains, s["in"]):
            _set(dm, f)
        s["batch"].run(0, 2)  # the first step plans, the second is captured: kept for the whole study
    elif kind == "heated":
        tab = heated_channel_table(4096, *HEATED_H_RANGE)
        col = _table_columns(tab)
        s["table"] = PropertyTable(tab, -1.0)
        s["dm"] = Domain(nc, **_channel_cfg(1.5, projection=PROJ_EXACT, precision=PREC_MIXED))
        s["in"] = _channel_fields(nc, 1.5, seed)
        yc = torch.from_numpy(_mesh_y(nc[1], 1.5)[1]).cuda()
        s["rhoh"] = _rhoh(0.8 + 0.35 * (yc * yc)[None, :, None] + 0.03 * _rand(4 * seed + 3, nc[2], nc[1], nc[0]), col)
        tw = float(np.interp(1.2, tab[:, 1], tab[:, 2]))
        s["dm"].thermo_enable(s["table"], (tw, tw), 1.0, float(np.interp(0.8, tab[:, 1], tab[:, 2])))
        s["cells"] = [torch.empty_like(s["rhoh"]) for _ in range(6)]
        s["g"] = [torch.empty_like(t) for t in s["in"][:3]]
    elif kind == "ops":
        s["dm"] = Domain(nc, **_channel_cfg(1.5, iacc=case["acc"]))
        s["in"] = _op_inputs(case, seed)
        s["out"] = [torch.empty(sh[2], sh[1], sh[0], device="cuda", dtype=s["in"][0].dtype)
                    for _, _, _, sh, _ in _operators(case)]
    elif kind == "poisson":
        s["dm"] = Domain(nc, **_channel_cfg(1.5))
        s["in"] = _poisson_rhs(case, seed)
        s["out"] = torch.empty_like(s["in"])
    elif kind == "props":
        tab = heated_channel_table(4096, *HEATED_H_RANGE)
        s["table"] = PropertyTable(tab, -1.0)
        if case["surrogate"]:
            s["sur"] = Surrogate(s["table"], nsamples=4096, seed=1)
            s["sur"].set_params(_surrogate_params(tab, s["sur"].info()[1].astype(np.float64), seed))
            s["table"].set_surrogate(s["sur"])
        s["in"] = _props_in(case, seed)
        s["out"] = [torch.empty_like(s["in"]) for _ in range(5 if case["surrogate"] else 7)]
    else:
        s["table"] = PropertyTable(heated_channel_table(4096, *HEATED_H_RANGE), -1.0)
        s["sur"] = Surrogate(s["table"], nsamples=1_000_000, seed=seed % (1 << 31))
    if "dm" in s and "out" not in s:
        s["out"] = [torch.empty_like(t) for t in s["in"]]
    if "batch" in s:
        s["out"] = [[torch.empty_like(t) for t in f] for f in s["in"]]
    torch.cuda.synchronize()
    return s


def _loop_projection(case):
    # the reference's single projection is only stable with the second-order scheme
    return PROJ_REFERENCE if case["acc"] == IACCU_CD2 else PROJ_EXACT


def _poisson_rhs(case, seed):
    r = _rand(seed, case["nz"], case["ny"], case["nx"])
    mc = torch.from_numpy(_mesh_y(case["ny"], 1.5)[3]).cuda()
    w = (1.0 / mc) / (1.0 / mc).sum()
    r -= (r.mean(dim=(0, 2)) * w).sum()  # the walls' compatibility: no net source
    return r.float() if case["f32"] else r


def _props_in(case, seed):
    col = _table_columns(heated_channel_table(4096, *HEATED_H_RANGE))
    return _rhoh(0.95 + 0.24 * _rand(seed, case["cells"]), col)


# What the mixed form keeps in single precision is read in single precision, as
# a program that writes such fields out or analyses them does.  Its pressure is
# an intermediate without an accuracy of its own (it carries the rounding of the
# right-hand side times dt^-1) and enters the velocities of every later sub-step;
# the velocities are the form's results.
def _mixed(fields):
    return [t.float() for t in fields[:3]]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("tgv", "channel"):
        _set(s["dm"], s["in"])
        s["dm"].run(0, case["steps"])
        _get(s["dm"], s["out"])
        return _mixed(s["out"]) if case.get("mixed") else s["out"]
    if kind == "loop":
        _set(s["dm"], s["in"])
        seen = []
        for it in range(case["steps"]):
            s["dm"].run(it, 1)
            mass = s["dm"].mass_check()
            rng = s["dm"].velocity_range()
            seen.append(rng)
        _get(s["dm"], s["out"])
        # (the windows' values are round-off: read as the loop reads them, not compared)
        return {"fields": s["out"], "range": np.stack(seen), "finite": int(np.isfinite(mass).all())}
    if kind == "batch":
        for dm, f in zip(s["batch"].domains, s["in"]):
            _set(dm, f)
        s["batch"].run(0, case["steps"])
        for dm, f in zip(s["batch"].domains, s["out"]):
            _get(dm, f)
        return [_mixed(f) for f in s["out"]]
    if kind == "heated":
        dm = s["dm"]
        _set(dm, s["in"])
        _lib.check(dm.lib.chs_thermo_set_rhoh(dm.h, _ptr(s["rhoh"]), _lib.MEM_DEVICE))
        dm.run(0, case["steps"])
        _get(dm, s["out"])
        _lib.check(dm.lib.chs_thermo_get(dm.h, *[_ptr(t) for t in s["cells"] + s["g"]], _lib.MEM_DEVICE))
        return _mixed(s["out"]) + [t.float() for t in s["cells"]]
    if kind == "ops":
        dm, (cell, node, wall) = s["dm"], s["in"]
        for (d, k, si, so, walls), out in zip(_operators(case), s["out"]):
            b = IBC_DIRICHLET if d == 1 else IBC_PERIODIC
            f = node if (d == 1 and k in (1, 5)) else cell
            args = (dm.h, d, k, case["acc"], _lib.ivec((b, b)), _ptr(f), _lib.ivec(si), _ptr(out), _lib.ivec(so),
                    _ptr(wall) if walls else None)
            _lib.check(dm.lib.chs_op3d_f32(*args) if case["f32"] else dm.lib.chs_op3d(*args, _lib.MEM_DEVICE))
        return s["out"]
    if kind == "poisson":
        s["out"].copy_(s["in"])
        L, h = s["dm"].lib, s["dm"].h
        _lib.check(L.chs_poisson_f32(h, _ptr(s["out"])) if case["f32"] else
                   L.chs_poisson(h, _ptr(s["out"]), _lib.MEM_DEVICE))
        return s["out"]
    if kind == "props":
        t = s["table"]
        outs = [_ptr(o) for o in s["out"]] + [None] * (7 - len(s["out"]))
        _lib.check(t.lib.chs_props_from_rhoh(t.h, _ptr(s["in"]), s["in"].numel(), *outs,
                                             PROPS_MLP if case["surrogate"] else PROPS_TABLE, _lib.MEM_DEVICE))
        return s["out"]
    loss = s["sur"].train(case["steps"], batch=case["batch"], lr=1e-3)
    return {"loss": np.float32(loss), "params": s["sur"].params()[0]}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("tgv", "loop", "channel", "heated"):
        n, steps = case["nx"] * case["ny"] * case["nz"], case["steps"]
        word = 4 if case.get("mixed") or kind == "heated" else 8
        return _flow_work(n, steps, word, kind == "heated")
    if kind == "batch":
        w = [_flow_work(g["nc"][0] * g["nc"][1] * g["nc"][2], case["steps"], 4, False) for g in _grids(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind == "ops":
        word = 4 if case["f32"] else 8
        n = [(si[0] * si[1] * si[2], so[0] * so[1] * so[2]) for _, _, si, so, _ in _operators(case)]
        return {"bytes": word * sum(a + b for a, b in n), "flops": 15 * sum(b for _, b in n)}
    if kind == "poisson":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 2 * n * (4 if case["f32"] else 8), "flops": n * _poisson_flops(n)}
    if kind == "props":
        n = case["cells"]
        return {"bytes": 8 * n * (6 if case["surrogate"] else 8), "flops": n * (2 * 2 * (64 + 64 * 64 + 64 * 5) if case["surrogate"] else 60)}
    return {"bytes": case["steps"] * (4 * 6 * case["batch"] + 4 * 7 * MLP_NP),
            "flops": case["steps"] * 3 * 2 * (64 + 64 * 64 + 64 * 5) * case["batch"]}


def _poisson_flops(n):
    return 5 * math.log2(n) + 15


def _flow_work(n, steps, word, heated):
    # per sub-step: velocity, pressure and the right-hand side kept from the last one, in
    # and out (FP64 state, the kept right-hand side in the form's precision), about 50
    # compact operators of 15 operations and the pressure solve
    bytes_ = 2 * (4 * 8 + 3 * word) + (2 * (8 + 8) + 4 * 8 if heated else 0)
    return {"bytes": 3 * steps * n * bytes_, "flops": 3 * steps * n * (50 * 15 + _poisson_flops(n))}


# --------------------------------------------------------------------------
# 64-bit values from dense operators
# --------------------------------------------------------------------------
# Interior schemes: (LHS off-diagonal, the two RHS weights) of the staggered first
# derivative and of the midpoint interpolation (Gaitonde & Visbal 1998).
def _scheme(deriv, acc):
    if deriv:
        al = {IACCU_CP4: 1 / 22, IACCU_CP6: 9 / 62}.get(acc, 0.0)
        a, b = {IACCU_CD2: (1.0, 0.0), IACCU_CP6: (63 / 62, 17 / 62)}.get(acc, ((9 - 6 * al) / 8, (-1 + 22 * al) / 8))
        return al, a, b / 3
    al = {IACCU_CP4: 1 / 6, IACCU_CP6: 3 / 10}.get(acc, 0.0)
    a, b = {IACCU_CD2: (1.0, 0.0), IACCU_CP6: (5 * (15 + 14 * al) / 64, (-25 + 126 * al) / 128)}.get(
        acc, (9 / 8 + 5 / 4 * al, -1 / 8 + 3 / 4 * al))
    return al, a / 2, b / 2


def _matrix(kind, n_in, acc, scale=1.0, walls=None):
    """Dense operator of one line: (M, W) with M (n_out x n_in) and W (n_out x 2) acting on the two wall values.
    kind: 0 / 1 interpolation to nodes / cells, 4 / 5 derivative to nodes / cells; walls: None periodic, "value"
    Dirichlet with wall values, "line" Dirichlet at a node of the line itself, "flux" zero wall gradient."""
    to_node, deriv = kind in (0, 4), kind >= 4
    sg = -1.0 if deriv else 1.0
    n = n_in if walls is None else (n_in + 1 if to_node else n_in - 1)
    rhs, lhs, wall = np.zeros((n, n_in)), np.eye(n), np.zeros((n, 2))
    near = (0, -1, 1, -2) if to_node else (1, 0, 2, -1)  # offsets of +c1, s c1, +c2, s c2

    def add(i, k, w):
        if walls is None:
            rhs[i, k % n_in] += w
        elif 0 <= k < n_in:
            rhs[i, k] += w
        else:  # ghost points: reflected about the wall
            side = 0 if k < 0 else 1
            edge = 0 if side == 0 else n_in - 1
            mirror = (-1 - k if side == 0 else 2 * n_in - 1 - k) if to_node else (-k if side == 0 else 2 * n_in - 2 - k)
            if walls == "flux":
                rhs[i, mirror] += w
            else:
                rhs[i, mirror] -= w
                if walls == "value":
                    wall[i, side] += 2 * w
                else:
                    rhs[i, edge] += 2 * w

    for i in range(n):
        end = walls is not None and i in (0, n - 1)
        if end and to_node and (walls == "flux" or not deriv):
            if walls == "value":
                wall[i, 0 if i == 0 else 1] = 1.0
            continue
        al, c1, c2 = _scheme(deriv, IACCU_CD4 if end and acc in (IACCU_CP4, IACCU_CP6) else acc)
        if al:
            lhs[i, (i - 1) % n] += al
            lhs[i, (i + 1) % n] += al
        for off, w in zip(near, (c1, sg * c1, c2, sg * c2)):
            add(i, i + off, w)
    m = np.linalg.solve(lhs, np.concatenate([rhs, wall], axis=1)) * (scale if deriv else 1.0)
    if not deriv or walls != "flux":
        return m[:, :n_in], m[:, n_in:]
    m[[0, -1]] = 0.0
    return m[:, :n_in], m[:, n_in:]


def _apply(m, f, d):
    """The matrix along x, y or z (0, 1, 2) of a (nz, ny, nx) tensor."""
    if d == 0:
        return f @ m.T
    if d == 1:
        return torch.stack([m @ p for p in f]) if f.shape[0] < 8 else torch.matmul(m, f)
    return (m @ f.reshape(f.shape[0], -1)).reshape(m.shape[0], *f.shape[1:])


class _Flow64:
    """The sub-step of the staggered solver with dense operators (constant properties)."""

    def __init__(self, nc, length, acc, dt, ren, beta=None):
        nx, ny, nz = nc
        self.dt, self.rre, self.walls = dt, 1.0 / ren, beta is not None
        h = [length[0] / nx, 1.0 / ny if self.walls else length[1] / ny, length[2] / nz]
        mp = mc = 1.0
        self.wy = torch.full((ny,), 1.0 / ny, dtype=torch.float64, device="cuda")
        if self.walls:
            mp, mc = (torch.from_numpy(v).cuda()[:, None] for v in _mesh_y(ny, beta)[2:])
            self.wy = (1.0 / mc[:, 0]) / (1.0 / mc[:, 0]).sum()
        dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
        self.m = {}
        for d, n in ((0, nx), (2, nz)) + (() if self.walls else ((1, ny),)):
            for k in (0, 1, 4, 5):
                self.m[d, k] = dev(_matrix(k, n, acc, 1.0 / h[d])[0])
        if self.walls:
            for name, k, w in (("value", 0, "value"), ("value", 4, "value"), ("value", 1, "value"), ("line", 5, "line"),
                               ("flux", 4, "flux")):
                m, e = _matrix(k, ny if k in (0, 4) else ny + 1, acc, 1.0 / h[1], w)
                f = (mp if k == 4 else mc) if k >= 4 else 1.0
                self.m[name, k], self.m[name, k, "w"] = dev(m) * f, dev(e) * f
            self.m[1, 0], self.m[1, 1] = self.m["value", 0], self.m["value", 1]
            self.m[1, 4], self.m[1, 5], grad = self.m["value", 4], self.m["line", 5], self.m["flux", 4]
        else:
            grad = self.m[1, 4]
        self.grad = {0: self.m[0, 4], 1: grad, 2: self.m[2, 4]}
        # D G: diagonal over kx, kz; eigen-decomposed along y
        self.lam = [torch.fft.fft((self.m[d, 5] @ self.m[d, 4])[:, 0]).real for d in (0, 2)]
        lam, v = np.linalg.eig((self.m[1, 5] @ grad).cpu().numpy())
        self.eig = dev(lam.astype(complex)), dev(v.astype(complex)), dev(np.linalg.inv(v.astype(complex)))

    def poisson(self, r, gauge_top=False):
        lam, v, vi = self.eig
        s = torch.matmul(vi, torch.fft.fft2(r, dim=(0, 2)))
        k = lam[None, :, None] + self.lam[0][None, None, :] + self.lam[1][:, None, None]
        null = int(lam.abs().argmin())
        k[0, null, 0] = 1.0
        s = s / k
        s[0, null, 0] = 0.0
        phi = torch.fft.ifft2(torch.matmul(v, s), dim=(0, 2)).real
        if gauge_top:
            phi = phi - phi[:, -1].mean()
        return phi

    def substep(self, q, p, old, sub, forced, gauge_top=False):
        A, m, r = _apply, self.m, self.rre
        tg, tz = (8 / 15, 5 / 12, 3 / 4)[sub], (0.0, -17 / 60, -5 / 12)[sub]
        ta, dt = tg + tz, self.dt
        to_c = [A(m[d, 1], q[d], d) for d in range(3)]  # each component at its cells
        dd = [A(m[d, 5], q[d], d) for d in range(3)]
        it = {(c, d): A(m[d, 0], q[c], d) for c in range(3) for d in range(3) if c != d}
        dv = {(c, d): A(m[d, 4], q[c], d) for c in range(3) for d in range(3) if c != d}
        div = dd[0] + dd[1] + dd[2]
        new = []
        for c in range(3):
            cur = 0.0
            for d in range(3):
                if c == d:
                    conv, visc = -to_c[c] * to_c[c], 2 * r * (dd[c] - div / 3)
                    cur = cur + A(m[d, 4], conv + visc, d)
                    if d == 1 and self.walls:
                        # wall values of the normal stress from the wall planes
                        dy = torch.matmul(m["value", 4][[0, -1]], to_c[1])
                        dx = A(m[0, 5], it[0, 1][:, [0, -1]], 0)
                        dz = A(m[2, 5], it[2, 1][:, [0, -1]], 2)
                        cur = cur + torch.matmul(m["value", 4, "w"], 2 * r * (dy - (dx + dy + dz) / 3))
                else:
                    a, b = (c, d) if c < d else (d, c)
                    cur = cur + A(m[d, 5], r * (dv[a, b] + dv[b, a]) - it[a, b] * it[b, a], d)
            rhs = dt * (tg * cur + (tz * old[c] if sub else 0.0) - ta * A(self.grad[c], p, c))
            if c == 0 and forced:
                rhs = rhs - (rhs.mean(dim=(0, 2)) * self.wy).sum()
            old[c] = cur
            new.append(q[c] + rhs)
        if self.walls:
            new[1][:, [0, -1]] = 0.0
        phi = self.poisson(sum(A(m[d, 5], new[d], d) for d in range(3)) / (ta * dt), gauge_top)
        new = [new[d] - dt * ta * A(self.grad[d], phi, d) for d in range(3)]
        if self.walls:
            new[1][:, [0, -1]] = 0.0
        return new, p + phi, old

    def step(self, q, p, forced, gauge_top=False):
        old = [0.0, 0.0, 0.0]
        for sub in range(3):
            q, p, old = self.substep(q, p, old, sub, forced, gauge_top)
        return q, p


def _exact_flow(flow, fields, steps, forced, gauge_top=False):
    q, p, seen = fields[:3], fields[3], []
    for _ in range(steps):
        q, p = flow.step(q, p, forced, gauge_top)
        seen.append([float(v) for t in q for v in (t.max(), t.min())])
    return q + [p], np.array(seen)


def exact(case, seed):
    kind = case["kind"]
    nc = (case.get("nx"), case.get("ny"), case.get("nz"))
    if kind == "tgv":
        p2 = 2 * math.pi
        return _exact_flow(_Flow64(nc, (p2, p2, p2), IACCU_CP6, 1e-3, 1600.0), _tgv_fields(nc, seed), case["steps"], False)[0]
    if kind == "loop":
        flow = _Flow64(nc, (LX, 2.0, LZ), case["acc"], DT, 2800.0, 1.5)
        f, seen = _exact_flow(flow, _channel_fields(nc, 1.5, seed), case["steps"], True, case["acc"] == IACCU_CD2)
        if case["acc"] != IACCU_CD2:
            f[3] = None  # the solve's gauge follows from its eigenvectors' scaling
        return {"fields": f, "range": seen, "finite": None}
    if kind == "channel":
        flow = _Flow64(nc, (LX, 2.0, LZ), IACCU_CP6, DT, 2800.0, case["beta"])
        f = _exact_flow(flow, _channel_fields(nc, case["beta"], seed), case["steps"], True)[0]
        return f[:3] if case["mixed"] else f[:3] + [None]
    if kind == "batch":
        return [_exact_flow(_Flow64(g["nc"], (LX, 2.0, LZ), IACCU_CP6, DT, g["ren"], g["beta"]),
                            _channel_fields(g["nc"], g["beta"], 100 * seed + i), case["steps"], True)[0][:3]
                for i, g in enumerate(_grids(case))]
    if kind == "ops":
        return _exact_ops(case, seed)
    if kind == "poisson":
        return _exact_poisson(case, seed)
    if kind == "props" and not case["surrogate"]:
        return _exact_props(case, seed)
    # heated: the whole coupled model; surrogate: BF16 weights and activations are part
    # of what it computes, so there is no value in 64 bits
    return None


def _exact_ops(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cell, node, wall = (t.double() for t in _op_inputs(case, seed))
    mp, mc = (torch.from_numpy(v).cuda()[:, None] for v in _mesh_y(ny, 1.5)[2:])
    out = []
    for d, k, si, so, walls in _operators(case):
        scale = (nx / LX, float(ny), nz / LZ)[d]
        m, w = _matrix(k, si[d], case["acc"], scale, None if d != 1 else ("value" if walls else "line"))
        m, w = torch.from_numpy(np.ascontiguousarray(m)).cuda(), torch.from_numpy(np.ascontiguousarray(w)).cuda()
        if d == 1 and k >= 4:
            m, w = m * (mp if k == 4 else mc), w * (mp if k == 4 else mc)
        f = _apply(m, node if (d == 1 and k in (1, 5)) else cell, d)
        out.append(f + torch.matmul(w, wall[:, :2]) if walls else f)
    return out


def _exact_poisson(case, seed):
    """FFT in x and z, the second-order y operator eliminated mode by mode; the mean mode's last unknown is zero."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    _, _, mp, mc = _mesh_y(ny, 1.5)
    lo, up = ny * ny * mc * mp[:-1], ny * ny * mc * mp[1:]
    lo[0] = up[-1] = 0.0
    s = torch.fft.rfft2(_poisson_rhs(case, seed).double(), dim=(0, 2))
    k = lambda n, l, m: -4 * (n / l) ** 2 * np.sin(np.pi * np.arange(m) / n) ** 2  # noqa: E731
    shift = torch.from_numpy(k(nz, LZ, nz)[:, None] + k(nx, LX, nx // 2 + 1)[None, :]).cuda()
    c = []
    for j in range(ny):
        b = shift - (lo[j] + up[j])
        if j:
            b = b - lo[j] * c[-1]
            s[:, j] -= lo[j] * s[:, j - 1]
        if j == ny - 1:
            b[0, 0] = 1.0
            s[0, j, 0] = 0.0
        c.append(up[j] / b)
        s[:, j] /= b
    for j in range(ny - 2, -1, -1):
        s[:, j] -= c[j] * s[:, j + 1]
    return torch.fft.irfft2(s, s=(nz, nx), dim=(0, 2))


def _exact_props(case, seed):
    col = _table_columns(heated_channel_table(4096, *HEATED_H_RANGE))
    tab = torch.from_numpy(heated_channel_table(4096, *HEATED_H_RANGE)).cuda()
    x, rh = _props_in(case, seed), (col["d"] * col["h"])
    h = _interp(x, rh.flip(0).contiguous(), col["h"].flip(0).contiguous())
    h = x / _interp(h, col["h"], col["d"])
    return [h] + [_interp(h, col["h"], c) for c in (col["d"], col["m"], col["k"], col["t"], tab[:, 7].contiguous(), col["cp"])]

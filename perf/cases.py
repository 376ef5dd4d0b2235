"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is a plain dict: its `kind` says which path of the framework it takes, the rest the sizes and options.

  conduction     the law d T = diffuse(k, T) through Solver.run, contracts off or judged every step
  black_scholes  a one-dimensional law on many lines (an option a plane)
  implicit       a law whose step solves tridiagonal systems along the lattice's lines
  valley         a many-term world law (12 fields, 14 terms), contracts every 8 steps
  heston         a batch of options of uneven lattices, every ADI step in one captured graph, then the prices
  rollout        the learned coarse lattice stepping (inference)
  train          a gradient and Adam step of the learned coarse lattice's net (backward)
  adjoint        the generated adjoint of a three-field law: states forward, then the sweep back over them
  mppi           a world model's planner: one plan for every agent
  nettrain       a world model's learn call: eight Adam steps on host rows, then the weights

Device inputs are torch tensors and device results are returned as torch views of the framework's own arrays.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "online-physics-cuda_amd"))

import field_hip  # noqa: E402

CONDUCTION_LAW = """field T init 0 range -1000000 1000000
param k = 0.1
term conduction
  d T = diffuse(k, T)
  conserves T
  max_dt = 0.15 * h * h / k
"""

BLACK_SCHOLES_LAW = """field V init 0 range -1 1000000
param sig = 0.2
param r = 0.05
term black_scholes
  d V = 0.5 * sig * sig * (shift(V, 1, 0, 0) - 2 * V + shift(V, -1, 0, 0)) / (h * h) + (r - 0.5 * sig * sig) * gx(V) - r * V
  max_dt = 0.4 * h * h / (sig * sig)
"""

IMPLICIT_X_LAW = """field T init 0 range -1000000 1000000
param k = 0.01
term crank_nicolson
  let a = 0.5 * k * dt / (h * h)
  d T = (tridiag_x(0 - a, 1 + 2 * a, 0 - a, T + a * (shift(T, 1, 0, 0) - 2 * T + shift(T, -1, 0, 0))) - T) / dt
"""

IMPLICIT_YZ_LAW = """field T init 0 range -1000000 1000000
field w init 1 range 0 10 static
param k = 0.05
term implicit_yz
  let a = k * w * dt / (h * h)
  let y1 = tridiag_y(0 - a, 1 + 2 * a, 0 - a, T)
  d T = (tridiag_z(0 - 0.5 * a, 1 + a, 0 - 0.5 * a, y1) - T) / dt
"""

VALLEY_FIELDS = ("rock", "sand", "water", "ice", "steam", "fuel", "flame", "smoke", "ash", "T", "wet", "near")
VALLEY_LAW = """field rock  init 0   range 0 1.01 static
field sand  init 0   range 0 1.01
field water init 0   range 0 1.01
field ice   init 0   range 0 1.01
field steam init 0   range 0 1.01
field fuel  init 0   range 0 1
field flame init 0   range 0 1.01 clamp
field smoke init 0   range 0 100 clamp
field ash   init 0   range 0 1.01
field T     init 290 range 0 8000
field wet   init 0   range 0 3
field near  init 0   range -1000 1000
derive wet = water + ice
derive wet += 0.5 * steam
derive near = distance(flame)

param g = 2.0
param k_rock = 0.6
param k_air = 0.05
param burn_at = 600
param burn_rate = 0.8
param heat_of_burning = 900

term settle
  let room = pos(1 - rock - sand - water - ice)
  d sand = fall(sand, rock + ice, g) + 0.2 * topple(sand, rock, 1)
  conserves sand
  max_dt = 0.4 * h / g

term pour
  d water = fall(water, rock + sand + ice, g) + spread(water, rock + sand + ice, 0.3) + 0.1 * topple(water, rock + sand, 1)
  conserves water
  max_dt = 0.4 * h / g

term conduct
  d T = diffuse(k_air + (k_rock - k_air) * (rock + sand + 0.5 * water), T)
  max_dt = 0.15 * h * h / k_rock

term burn
  let hot = step(T - burn_at)
  let rate = burn_rate * min(fuel, hot * (0.2 + flame))
  d fuel = -rate
  d flame = 2 * rate - 0.5 * flame * step(0.05 - fuel)
  d T = heat_of_burning * rate
  d ash = 0.3 * rate

term catch
  let neighbours = max(max(shift(flame, 1, 0, 0), shift(flame, -1, 0, 0)), max(shift(flame, 0, 1, 0), shift(flame, 0, -1, 0)))
  d flame = 0.5 * fuel * step(neighbours - 0.3) * step(T - 450)

term rise
  d smoke = 0.6 * flame - 0.3 * gz(smoke) - 0.02 * smoke + 0.05 * lap(smoke)
  d T = -0.1 * adv(T, 0, 0, 0.4 * flame)

term freeze
  let cold = step(273 - T)
  d ice = 0.5 * water * cold - 0.5 * ice * step(T - 273)
  d water = -0.5 * water * cold + 0.5 * ice * step(T - 273)
  conserves water + ice

term boil
  let boiling = pos(T - 373) / 100
  d steam = 0.4 * min(water, boiling) - 0.05 * steam * step(350 - T)
  d water = -0.4 * min(water, boiling) + 0.05 * steam * step(350 - T)
  d T = -40 * min(water, boiling)

term vapour
  d steam = -0.5 * gz(steam) + 0.1 * lap(steam) + 0.01 * (shift(steam, 0, 0, -1) - steam)

term wind
  d smoke = 0.05 * (maxof(T) - T) / (maxof(T) + 1) * gx(smoke) + 0.02 * gy(smoke)

term radiate
  d T = -0.0002 * pos(T - 290) * (1 - rock) + 0.01 * sqrt(pos(T - 290)) * step(0.5 - near)

term press
  d water = 0.0005 * poisson(wet - 0.4, 8) * (1 - rock)

term crumble
  d sand = 0.02 * rock * step(T - 1200) * (1 - sand)

term cool_ash
  d ash = -0.01 * ash * step(350 - T) + 0.005 * max(shift(ash, 0, 0, 1) - ash, 0)
"""

TRANSPORT_LAW = """field a init 0
field b init 0
field c init 0
param Da = 0.05
param Db = 0.02
param Dc = 0.01
term transport
  d a = diffuse(Da, a) - 0.3 * (a - shift(a, -1, 0, 0)) / h + 0.2 * (shift(a, 0, 1, 0) - a) / h - 0.1 * (a - shift(a, 0, 0, -1)) / h - a * b + 0.1 * c
  d b = diffuse(Db, b) - 0.3 * (b - shift(b, -1, 0, 0)) / h + 0.2 * (shift(b, 0, 1, 0) - b) / h - 0.1 * (b - shift(b, 0, 0, -1)) / h - a * b + 0.1 * c
  d c = diffuse(Dc, c) - 0.3 * (c - shift(c, -1, 0, 0)) / h + 0.2 * (shift(c, 0, 1, 0) - c) / h - 0.1 * (c - shift(c, 0, 0, -1)) / h + a * b - 0.1 * c
"""


def listed():
    return [
        # The smallest lattice the tests and the refinement study run: launches and latency are all of it.
        {"name": "conduction_32", "kind": "conduction", "nx": 32, "ny": 32, "nz": 32, "steps": 64, "judged": False},
        # The headline lattice, stepped as a simulation runs it.
        {"name": "conduction_256", "kind": "conduction", "nx": 256, "ny": 256, "nz": 256, "steps": 32, "judged": False},
        # A large lattice of odd sizes with the contracts judged every step, as a run that must not break them is taken.
        {"name": "conduction_odd_judged", "kind": "conduction", "nx": 501, "ny": 333, "nz": 290, "steps": 4, "judged": True},
        # Options priced by the law, 512 lines of 4096 cells.
        {"name": "black_scholes_4096", "kind": "black_scholes", "nx": 4096, "nz": 512, "steps": 32},
        # Implicit steps along y and z with a field-dependent operator.
        {"name": "implicit_yz_256", "kind": "implicit", "axis": "yz", "nx": 256, "ny": 256, "nz": 256, "steps": 4},
        # A world of a million cells over two seconds of play.
        {"name": "valley_144", "kind": "valley", "nx": 144, "ny": 144, "nz": 48, "steps": 8},
        # A book of 2048 options of three lattice sizes.
        {"name": "heston_2048", "kind": "heston", "options": 2048, "steps": 64, "scheme": 0, "ragged": False},
        # Four unseen starts of the learned coarse lattice, a quarter of a run.
        {"name": "rollout_128", "kind": "rollout", "n": 128, "count": 4, "steps": 25},
        # One training step on a batch of sixteen coarse lattices.
        {"name": "train_128", "kind": "train", "n": 128, "count": 16},
        # A segment of reverse mode: eight states kept, eight adjoint steps back over them.
        {"name": "adjoint_256", "kind": "adjoint", "nx": 256, "ny": 256, "nz": 256, "steps": 8},
        # The planner for a crowd of agents.
        {"name": "mppi_256", "kind": "mppi", "agents": 256, "samples": 512, "horizon": 32, "features": 16, "hidden": 64},
        # The world model's own learn call: 1024 rows, host memory in and out.
        {"name": "nettrain_1024", "kind": "nettrain", "rows": 1024, "features": 16, "hidden": 64, "act": "tanh"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("conduction", "conduction", "black_scholes", "implicit", "valley", "heston", "rollout", "train", "adjoint", "mppi", "nettrain"))
    if kind == "conduction":
        nx, ny, nz = (_log(rng, 16, 512) for _ in range(3))
        if rng.random() < 0.6:
            nx = (nx + 3) // 4 * 4  # rows of whole 16-byte quads are what most programs choose
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "steps": rng.randint(2, 32), "judged": rng.random() < 0.4}
    if kind == "black_scholes":
        return {"kind": kind, "nx": _log(rng, 64, 4096), "nz": _log(rng, 1, 512), "steps": rng.randint(2, 32)}
    if kind == "implicit":
        nx, ny, nz = (_log(rng, 16, 320) for _ in range(3))
        return {"kind": kind, "axis": rng.choice(("x", "yz")), "nx": nx, "ny": ny, "nz": nz, "steps": rng.randint(1, 8)}
    if kind == "valley":
        return {"kind": kind, "nx": _log(rng, 32, 160), "ny": _log(rng, 32, 144), "nz": _log(rng, 16, 64), "steps": rng.randint(2, 12)}
    if kind == "heston":
        return {"kind": kind, "options": _log(rng, 4, 2048), "steps": _log(rng, 16, 64), "scheme": rng.choice((0, 0, 1)), "ragged": rng.random() < 0.5}
    if kind == "rollout":
        return {"kind": kind, "n": _log(rng, 32, 256), "count": _log(rng, 1, 32), "steps": rng.randint(2, 25)}
    if kind == "train":
        return {"kind": kind, "n": _log(rng, 32, 160), "count": _log(rng, 1, 16)}
    if kind == "adjoint":
        nx, ny, nz = (_log(rng, 16, 256) for _ in range(3))
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "steps": rng.randint(2, 8)}
    if kind == "mppi":
        return {"kind": kind, "agents": _log(rng, 1, 256), "samples": 16 * _log(rng, 2, 32), "horizon": rng.randint(8, 32),
                "features": rng.randint(4, 24), "hidden": 16 * rng.randint(1, 6)}
    return {"kind": kind, "rows": _log(rng, 64, 65536), "features": rng.randint(4, 24), "hidden": rng.randint(16, 96),
            "act": rng.choice(("tanh", "tanh", "relu", "silu", "gelu"))}


# ---- inputs, made from the seed alone ----


def _uniform(n, seed, lo=0.0, hi=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _normal(shape, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _payoff(nx, nz, seed):
    """Puts of strikes about 100 on x = ln S in ln 100 +- 4, averaged over each cell, a strike a plane."""
    h = 8.0 / nx
    edges = math.log(100.0) - 4.0 + h * torch.arange(nx + 1, device="cuda", dtype=torch.float64)
    lo, hi = edges[:-1], edges[1:]
    strike = _uniform(nz, seed, 80.0, 120.0).double()[:, None]
    top = torch.minimum(hi, torch.log(strike))
    pay = torch.where(top > lo, (strike * (top - lo) - (torch.exp(top) - torch.exp(lo))) / h, torch.zeros((), device="cuda", dtype=torch.float64))
    return pay.float().reshape(-1).contiguous()


def _valley(case, seed):
    """A rock floor, a sand bank, fuel with a fire in it, a pond and ice, in proportion to the lattice."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    z, y, x = torch.meshgrid(torch.arange(nz, device="cuda") * (24.0 / nz), torch.arange(ny, device="cuda") * (40.0 / ny),
                             torch.arange(nx, device="cuda") * (48.0 / nx), indexing="ij")
    ball = (x - 20) ** 2 + (y - 20) ** 2 + (z - 7) ** 2
    ice = ((z >= 5) & (z < 7) & (x >= 40) & (y >= 30)).float()
    t = torch.full_like(x, 290.0)
    t = torch.where(ball <= 9, torch.full_like(x, 1400.0), t)
    t = torch.where(ice > 0, torch.full_like(x, 250.0), t)
    zero = torch.zeros_like(x)
    fields = {"rock": (z < 5).float(), "sand": ((z >= 5) & (z < 7) & (x < 20)).float(),
              "water": ((z >= 5) & (z < 10) & (x >= 34) & (x < 44) & (y >= 4) & (y < 14)).float(), "ice": ice, "steam": zero,
              "fuel": ((z >= 5) & (z < 8) & (x >= 12) & (x < 30) & (y >= 10) & (y < 30)).float(),
              "flame": torch.where(ball <= 4, torch.full_like(x, 0.6), zero), "smoke": zero, "ash": zero,
              "T": t + 0.5 * _uniform(nx * ny * nz, seed).reshape(nz, ny, nx)}
    return {k: v.float().reshape(-1).contiguous() for k, v in fields.items()}


def _options(case, seed):
    """nx, ny and the eight numbers of each option: three lattice sizes, a third each; ragged: any row count below."""
    rng = np.random.default_rng(seed)
    n = case["options"]
    shapes = ((128, 64), (256, 128), (512, 256))
    pick = rng.integers(0, 3, n)
    nx = np.array([shapes[i][0] for i in pick], np.int32)
    ny = np.array([shapes[i][1] for i in pick], np.int32)
    if case["ragged"]:
        ny = np.array([rng.integers(v // 2 + 1, v + 1) for v in ny], np.int32)
    opts = np.stack([rng.uniform(0.5, 5, n), rng.uniform(0.01, 0.1, n), rng.uniform(0.1, 0.8, n), rng.uniform(-0.9, -0.1, n),
                     np.full(n, 0.02), rng.uniform(80, 120, n), rng.uniform(0.25, 2, n), rng.uniform(0.01, 0.1, n)], 1)
    return nx, ny, opts


HESTON_THETA = (0.5, 0.5 + math.sqrt(3.0) / 6.0)  # Craig-Sneyd, Hundsdorfer-Verwer
COARSE = {"du": 1e-3, "dv": 5e-3, "k": 5e-3, "scale": 0.325}


def _coarse_net(seed):
    rng = np.random.default_rng(seed)
    parts = []
    for fan_in, fan_out, size in ((18, 64, 1.0), (64, 64, 1.0), (64, 2, 0.2)):
        lim = math.sqrt(6.0 / (fan_in + fan_out)) * size
        parts += [rng.uniform(-lim, lim, (fan_in, fan_out)).reshape(-1), rng.uniform(-0.05, 0.05, fan_out)]
    return np.concatenate(parts).astype(np.float32)


def _coarse_dt(n):
    return 8e-3 * min(1.0, (128.0 / n) ** 2)


def _coarse_lap(f, h):
    p = torch.cat([f[:, :, :1], f, f[:, :, -1:]], 2)
    q = torch.cat([f[:, :1], f, f[:, -1:]], 1)
    return (p[:, :, 2:] + p[:, :, :-2] + q[:, 2:] + q[:, :-2] - 4 * f) / (h * h)


def _coarse_rates(u, v, h):
    return (COARSE["du"] * _coarse_lap(u, h) + u - u ** 3 - COARSE["k"] - v, COARSE["dv"] * _coarse_lap(v, h) + u - v)


def _coarse_states(case, seed):
    """A start of N(0, 1) cells relaxed by the law for a few steps, as a run's snapshots are."""
    n, count = case["n"], case["count"]
    h, dt = 2.0 / n, _coarse_dt(n)
    u, v = _normal((count, n, n), 2 * seed).double(), _normal((count, n, n), 2 * seed + 1).double()
    for _ in range(4):
        ru, rv = _coarse_rates(u, v, h)
        u, v = u + dt * ru, v + dt * rv
    return u.float().contiguous(), v.float().contiguous()


def _world_net(case, seed):
    """Dynamics weights (.net layout): features + 2 -> hidden -> hidden -> features, about unit gain."""
    F, hid = case["features"], case["hidden"]
    rng = np.random.default_rng(seed)
    sizes = [F + 2, hid, hid, F]
    parts = []
    for k, gain in zip(range(3), (1.0, 1.0, 0.5)):
        parts += [(rng.uniform(-1, 1, (sizes[k + 1], sizes[k])) * gain * math.sqrt(3.0 / sizes[k])).reshape(-1), rng.uniform(-0.1, 0.1, sizes[k + 1])]
    return sizes, np.concatenate(parts).astype(np.float32), rng


def _plan_inputs(case, seed):
    sizes, flat, rng = _world_net(case, seed)
    F = case["features"]
    return {"sizes": sizes, "flat": flat, "target": rng.uniform(-0.5, 0.5, F).astype(np.float32),
            "obs": rng.uniform(-1, 1, (case["agents"], F)).astype(np.float32), "ids": np.arange(case["agents"], dtype=np.uint32),
            "mean": rng.uniform(-0.3, 0.3, (case["agents"], case["horizon"], 2)).astype(np.float32), "tick": 1 + seed % 1000}


def _learn_inputs(case, seed):
    sizes, flat, rng = _world_net(case, seed)
    F = case["features"]
    head = np.concatenate([rng.uniform(-0.1, 0.1, F + 2), rng.uniform(0.8, 1.2, F + 2), [0.9]]).astype(np.float32)
    image = np.concatenate([head, np.zeros(-head.size % 4, np.float32), flat])
    x = rng.uniform(-1, 1, (case["rows"], F + 2)).astype(np.float32)
    mix = rng.uniform(-1, 1, (F, F + 2)) / math.sqrt(F + 2)
    return sizes, image, x, np.sin(x @ mix.T).astype(np.float32)


# ---- what a program has in hand before the call ----


class _Memory:
    """A device array of the framework's as torch takes it."""

    def __init__(self, owner, ptr, count, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": kind, "data": (ptr, False), "version": 2, "strides": None}


def _view(state, owner, ptr, count, kind="<f4"):
    """The torch view of a device array (a field's two arrays come in turn, so the views are kept by address). A view
    keeps the object that owns the array alive, also after the state is gone."""
    views = state.setdefault("views", {})
    if ptr not in views:
        views[ptr] = torch.as_tensor(_Memory(owner, ptr, count, kind), device="cuda")
        views[ptr].owner = owner
    return views[ptr]


def _solver(law, shape, h, every, fields, dt):
    s = field_hip.Solver(law, shape, h)
    s.set_lazy_readback(True)
    s.check_contracts_every(every)
    s.refresh_derived()  # the declared start goes up; from here on the fields are written on the card
    torch.cuda.synchronize()
    for name, v in fields.items():
        s.set_field_device(name, v.data_ptr())
    s.step(dt)
    field_hip.sync()
    return s


def _conduction_dt(case):
    h = 1.0 / max(case["nx"], case["ny"], case["nz"])
    return h, 0.4 * h * h / 0.1 / 3


def prepare(case, seed):
    kind = case["kind"]
    if kind == "conduction":
        cells = case["nx"] * case["ny"] * case["nz"]
        h, dt = _conduction_dt(case)
        start = {"T": _uniform(cells, seed)}
        law = field_hip.Law(CONDUCTION_LAW)
        s = _solver(law, (case["nx"], case["ny"], case["nz"]), h, 1 if case["judged"] else 1 << 30, start, dt)
        return {"case": case, "solver": s, "start": start, "out": ("T",), "dt": dt, "cells": cells}
    if kind == "black_scholes":
        cells = case["nx"] * case["nz"]
        h = 8.0 / case["nx"]
        dt = 0.4 * h * h / (0.2 * 0.2)
        start = {"V": _payoff(case["nx"], case["nz"], seed)}
        s = _solver(field_hip.Law(BLACK_SCHOLES_LAW), (case["nx"], 1, case["nz"]), h, 1 << 30, start, dt)
        return {"case": case, "solver": s, "start": start, "out": ("V",), "dt": dt, "cells": cells}
    if kind == "implicit":
        cells = case["nx"] * case["ny"] * case["nz"]
        h = 1.0 / max(case["nx"], case["ny"], case["nz"])
        start = {"T": _uniform(cells, 2 * seed)}
        if case["axis"] == "x":
            law, dt = field_hip.Law(IMPLICIT_X_LAW), 0.5 * h * h / 0.01
            s = _solver(law, (case["nx"], case["ny"], case["nz"]), h, 1 << 30, start, dt)
        else:
            law, dt = field_hip.Law(IMPLICIT_YZ_LAW), 0.5 * h * h / 0.05
            w = _uniform(cells, 2 * seed + 1, 0.5, 2.0)
            s = _solver(law, (case["nx"], case["ny"], case["nz"]), h, 1 << 30, dict(start, w=w), dt)
        return {"case": case, "solver": s, "start": start, "out": ("T",), "dt": dt, "cells": cells}
    if kind == "valley":
        cells = case["nx"] * case["ny"] * case["nz"]
        start = _valley(case, seed)
        s = _solver(field_hip.Law(VALLEY_LAW), (case["nx"], case["ny"], case["nz"]), 0.5, 8, start, 0.25)
        return {"case": case, "solver": s, "start": start, "out": VALLEY_FIELDS, "dt": 0.25, "cells": cells}
    if kind == "heston":
        nx, ny, opts = _options(case, seed)
        b = field_hip.HestonBatch(nx, ny, opts, case["steps"], case["scheme"], HESTON_THETA[case["scheme"]])
        b.tune(2)
        b.capture(case["steps"])
        b.sync()
        return {"case": case, "batch": b, "largest": int(np.argmax(nx.astype(np.int64) * ny))}
    if kind == "rollout":
        u, v = _coarse_states(case, seed)
        net = field_hip.LearnedNet(_coarse_net(seed), COARSE["scale"])
        torch.cuda.synchronize()
        return {"case": case, "net": net, "u": u, "v": v, "bufs": [torch.empty_like(u) for _ in range(4)]}
    if kind == "train":
        u, v = _coarse_states(case, seed)
        n = case["n"]
        h, dt = 2.0 / n, _coarse_dt(n)
        ru, rv = _coarse_rates(u.double(), v.double(), h)
        u1 = (u.double() + dt * (ru + 0.3 * _normal(u.shape, seed + 7).double())).float().contiguous()
        v1 = (v.double() + dt * (rv + 0.3 * _normal(u.shape, seed + 8).double())).float().contiguous()
        net = field_hip.LearnedNet(_coarse_net(seed), COARSE["scale"])
        torch.cuda.synchronize()
        return {"case": case, "net": net, "u": u, "v": v, "u1": u1, "v1": v1}
    if kind == "adjoint":
        shape = (case["nx"], case["ny"], case["nz"])
        cells = shape[0] * shape[1] * shape[2]
        h, dt = _transport_dt(case)
        law = field_hip.Law(TRANSPORT_LAW)
        adj_law = field_hip.Law(law.adjoint("transport"))
        start = {f: _uniform(cells, 4 * seed + i, 0.2, 1.0) for i, f in enumerate("abc")}
        primal = _solver(law, shape, h, 1 << 30, start, dt)
        adj = _solver(adj_law, shape, h, 1 << 30, {}, dt)
        ring = [{f: field_hip.DeviceArray(cells) for f in "abc"} for _ in range(case["steps"])]
        sums = {p: field_hip.DeviceArray(4) for p in ("Da", "Db", "Dc")}
        seed_c = _normal((cells,), 4 * seed + 3)
        torch.cuda.synchronize()
        return {"case": case, "primal": primal, "adj": adj, "start": start, "seed": seed_c, "ring": ring, "sums": sums, "dt": dt, "cells": cells}
    if kind == "mppi":
        q = _plan_inputs(case, seed)
        F = case["features"]
        pl = field_hip.MppiPlanner(F, case["hidden"], case["horizon"], case["samples"])
        pl.set_dynamics(q["flat"], np.zeros(F + 2, np.float32), np.ones(F + 2, np.float32), np.ones(F, np.float32))
        pl.set_cost(q["target"], np.ones(F, np.float32), 0.01)
        return {"case": case, "planner": pl, "inputs": q}
    sizes, image, x, t = _learn_inputs(case, seed)
    tr = field_hip.NetTrainer(sizes, case["act"])
    tr.set_image(image)
    return {"case": case, "trainer": tr, "x": x, "t": t}


def _transport_dt(case):
    h = 1.0 / max(case["nx"], case["ny"], case["nz"])
    return h, 0.8 * h * h / (6 * 0.05)


# ---- one pass ----


def run(state):
    case = state["case"]
    kind = case["kind"]
    if "solver" in state:
        s = state["solver"]
        for name, v in state["start"].items():
            s.set_field_device(name, v.data_ptr())
        s.run(state["dt"], case["steps"])
        out = [_view(state, s, s.field_device(name), state["cells"]) for name in state["out"]]
        if case.get("judged"):
            out.append(len(s.violations()))
        return out
    if kind == "heston":
        b = state["batch"]
        b.reset()
        b.launch()
        return b.prices(), b.lattice(state["largest"])
    if kind == "rollout":
        n, count = case["n"], case["count"]
        cur, bufs = (state["u"], state["v"]), state["bufs"]
        for i in range(case["steps"]):
            nxt = (bufs[2 * (i % 2)], bufs[2 * (i % 2) + 1])
            state["net"].step(cur[0].data_ptr(), cur[1].data_ptr(), n, n, count, 2.0 / n, COARSE["du"], COARSE["dv"], COARSE["k"],
                              _coarse_dt(n), nxt[0].data_ptr(), nxt[1].data_ptr(), learned=True, bound=50.0)
            cur = nxt
        return cur
    if kind == "train":
        n = case["n"]
        loss, g = state["net"].gradient(state["u"].data_ptr(), state["v"].data_ptr(), state["u1"].data_ptr(), state["v1"].data_ptr(), n, n,
                                        case["count"], 2.0 / n, COARSE["du"], COARSE["dv"], COARSE["k"], _coarse_dt(n))
        state["net"].adam(1e-3)
        return loss, g
    if kind == "adjoint":
        return _adjoint_pass(state)
    if kind == "mppi":
        q = state["inputs"]
        return state["planner"].plan(q["obs"], q["ids"], q["mean"], q["tick"], 0.3, 0.1)[0]
    tr = state["trainer"]
    losses = [tr.step(state["x"], state["t"]) for _ in range(8)]
    return losses, tr.image()


def _adjoint_pass(state):
    """The vector-Jacobian product of the run: states kept forward, the adjoint law stepped back over them."""
    lib, check = field_hip.lib(), field_hip.check
    primal, adj, ring, dt, cells = state["primal"], state["adj"], state["ring"], state["dt"], state["cells"]
    for f in "abc":
        primal.set_field_device(f, state["start"][f].data_ptr())
    for j, slot in enumerate(ring):
        for f in "abc":
            check(lib.fe_hip_memcpy_dtod_async(slot[f].ptr, primal.field_device(f), 4 * cells), "save")
        if j + 1 < len(ring):
            primal.step(dt)
    for f in "ab":
        adj.fill_field(f + "__adj", 0.0)
    adj.set_field_device("c__adj", state["seed"].data_ptr())
    for p, acc in state["sums"].items():
        adj.fill_field(p + "__adj", 0.0)
        check(lib.fe_hip_memset_d32_async(acc.ptr, 0, 4), "clear")
    for slot in reversed(ring):
        for f in "abc":
            adj.bind_field_device(f, slot[f])
        adj.step(dt)
        for p, acc in state["sums"].items():
            adj.total_accumulate(p + "__adj", acc)
            adj.fill_field(p + "__adj", 0.0)
    grads = [_view(state, adj, adj.field_device(f + "__adj"), cells) for f in "abc"]
    return grads, [_view(state, acc, acc.ptr, 1, "<f8") for acc in state["sums"].values()]


# ---- what a pass cannot do without ----


def work(case):
    kind = case["kind"]
    if kind == "conduction":
        c = case["nx"] * case["ny"] * case["nz"] * case["steps"]
        return {"bytes": 8.0 * c, "flops": 15.0 * c}
    if kind == "black_scholes":
        c = case["nx"] * case["nz"] * case["steps"]
        return {"bytes": 8.0 * c, "flops": 16.0 * c}
    if kind == "implicit":
        c = case["nx"] * case["ny"] * case["nz"] * case["steps"]
        return {"bytes": (8.0 if case["axis"] == "x" else 12.0) * c, "flops": (18.0 if case["axis"] == "x" else 30.0) * c}
    if kind == "valley":  # 12 fields read, the 11 that change written
        c = case["nx"] * case["ny"] * case["nz"] * case["steps"]
        return {"bytes": 92.0 * c, "flops": 400.0 * c}
    if kind == "heston":  # the lattice read and written once a step
        c = case["options"] * (128 * 64 + 256 * 128 + 512 * 256) / 3.0 * (0.75 if case["ragged"] else 1.0) * case["steps"]
        return {"bytes": 8.0 * c, "flops": 60.0 * c}
    if kind in ("rollout", "train"):  # four evaluations of the net a cell; backward twice as much again
        c = case["n"] * case["n"] * case["count"] * case.get("steps", 1)
        return {"bytes": 16.0 * c, "flops": 4 * 10752.0 * c * (3 if kind == "train" else 1)}
    if kind == "adjoint":  # forward: three fields read and written; back: nine read, six written
        c = case["nx"] * case["ny"] * case["nz"] * case["steps"]
        return {"bytes": 84.0 * c, "flops": 300.0 * c}
    F, hid = case["features"], case["hidden"]
    products = (F + 2) * hid + hid * hid + hid * F
    if kind == "mppi":
        futures = case["agents"] * case["samples"]
        return {"bytes": 4.0 * (case["agents"] * (F + 4 * case["horizon"]) + products), "flops": 2.0 * futures * case["horizon"] * products}
    return {"bytes": 4.0 * (case["rows"] * (2 * F + 2) * 8 + 2 * products), "flops": 8 * 2.0 * case["rows"] * (3 * products - (F + 2) * hid)}


def tolerance(case):
    """Four times the largest error seen against exact(), which a correct path at the same precision can show too."""
    kind = case["kind"]
    if kind in ("conduction", "black_scholes", "implicit", "valley"):
        return "exact"  # the engine gives its reference's bits
    if kind == "heston":
        return {"rel": 4e-7}
    if kind == "rollout":
        return {"rel": 1e-3}  # bf16 weights and activations
    if kind == "train":
        return {"rel": 2e-2}
    if kind == "adjoint":
        return {"rel": 1.3e-5}  # a diffusivity's total cancels; the fields' gradients are within 1e-7
    if kind == "mppi":
        return {"rel": 3e-3}  # fp16 products
    return {"rel": 3e-6}


# ---- the same outputs in 64 bits ----


def _shift(f, axis, by):
    """f at the next cell along `axis` (by = 1) or the one before (-1), the edge cell repeating."""
    n = f.shape[axis]
    body = f.narrow(axis, 1, n - 1) if by > 0 else f.narrow(axis, 0, n - 1)
    edge = f.narrow(axis, n - 1, 1) if by > 0 else f.narrow(axis, 0, 1)
    return torch.cat([body, edge] if by > 0 else [edge, body], axis)


def _diffuse(f, k, h):
    total = -6 * f
    for axis in range(3):
        total = total + _shift(f, axis, 1) + _shift(f, axis, -1)
    return k * total / (h * h)


def _line_solve(a, b, c, d, axis):
    """Tridiagonal systems along `axis`, the edge cell repeating past the ends."""
    a, b, c, d = (torch.movedim(v.expand_as(d) if torch.is_tensor(v) else torch.full_like(d, v), axis, 0).contiguous() for v in (a, b, c, d))
    b = b.clone()
    b[0] += a[0]
    b[-1] += c[-1]
    n = d.shape[0]
    m, y = torch.empty_like(d), torch.empty_like(d)
    for i in range(n):
        piv = b[i] - a[i] * m[i - 1] if i else b[i]
        m[i] = c[i] / piv
        y[i] = ((d[i] - a[i] * y[i - 1]) if i else d[i]) / piv
    for i in range(n - 2, -1, -1):
        y[i] -= m[i] * y[i + 1]
    return torch.movedim(y, 0, axis)


def _heston_exact(case, seed):
    nx, ny, opts = _options(case, seed)
    n, steps, scheme = case["options"], case["steps"], case["scheme"]
    theta = HESTON_THETA[scheme]
    prices = np.empty(n)
    largest = int(np.argmax(nx.astype(np.int64) * ny))
    lattice = None
    groups = {}
    for o in range(n):
        groups.setdefault((int(nx[o]), int(ny[o])), []).append(o)
    if len(groups) * steps > 600:
        return None  # every row count its own group: over the time an exact answer may take
    for (X, Y), members in groups.items():
        P = torch.tensor(opts[members], device="cuda", dtype=torch.float64)
        kappa, th, sig, rho, r, strike, mat, _ = (P[:, i, None, None] for i in range(8))
        h = 6.0 / X
        dt = mat / steps
        j = torch.arange(Y, device="cuda", dtype=torch.float64)[None, :, None]
        var = sig * (j + 0.5) * h
        e0 = (j == 0).double()
        drift = kappa * (th - var) / sig - 0.5 * sig
        lx = 0.5 * var / h ** 2 - (r - 0.5 * var) / (2 * h)
        ux = 0.5 * var / h ** 2 + (r - 0.5 * var) / (2 * h)
        ly = 0.5 * (var - 0.5 * sig * h) / h ** 2 - (1 - e0) * drift / (2 * h)
        uy = 0.5 * (var + 0.5 * sig * h) / h ** 2 + (1 + e0) * drift / (2 * h)

        def factor(low, up, count, line):
            a, c = -theta * dt * low, -theta * dt * up
            b = 1.0 + theta * dt * (low + up + 0.5 * r)
            ms, inv = [], []
            for i in range(count):
                ai, bi, ci = (v[:, i] if line else v[:, :, 0] for v in (a, b, c))
                bi = bi + (ai if i == 0 else 0.0) + (ci if i + 1 == count else 0.0)
                piv = bi - ai * ms[-1] if i else bi
                inv.append(1.0 / piv)
                ms.append(ci / piv)
            return a, ms, inv

        def solve(f, d, line):
            a, ms, inv = f
            y = d.movedim(1 if line else 2, 0).contiguous()
            for i in range(len(ms)):
                ai = a[:, i] if line else a[:, :, 0]
                y[i] = (torch.addcmul(y[i], ai, y[i - 1], value=-1) if i else y[i]) * inv[i]
            for i in range(len(ms) - 2, -1, -1):
                y[i].addcmul_(ms[i].expand_as(y[i]), y[i + 1], value=-1)
            return y.movedim(0, 1 if line else 2)

        fx, fy = factor(lx, ux, X, False), factor(ly, uy, Y, True)

        def mixed(w):
            g = (_shift(w, 1, 1) - _shift(w, 1, -1)) / (2 * h)
            g[:, 0] *= 2
            g[:, -1] *= 2
            g = (_shift(g, 2, 1) - _shift(g, 2, -1)) / (2 * h)
            g[:, :, 0] *= 2
            g[:, :, -1] *= 2
            return rho * var * g

        def full(w):
            return (mixed(w) + lx * (_shift(w, 2, -1) - w) + ux * (_shift(w, 2, 1) - w) + ly * (_shift(w, 1, -1) - w)
                    + uy * (_shift(w, 1, 1) - w) - r * w)

        x = math.log(100.0) - 3.0 + (torch.arange(X, device="cuda", dtype=torch.float64) + 0.5) * h
        lk = torch.log(strike)
        lo, hi = torch.minimum(x - 0.5 * h, lk), torch.minimum(x + 0.5 * h, lk)
        U = ((strike * (hi - lo) - (torch.exp(hi) - torch.exp(lo))) / h).expand(len(members), Y, X).contiguous()
        for _ in range(steps):
            fu = full(U)
            d2 = solve(fy, solve(fx, dt * fu, False), True)
            second = 0.5 * dt * mixed(d2) if scheme == 0 else dt * fu - d2 + 0.5 * dt * full(d2)
            U = U + (d2 + solve(fy, solve(fx, second, False), True))
        U = U.cpu().numpy()
        for q, o in enumerate(members):
            tx = 3.0 / h - 0.5
            ty = (opts[o, 7] / opts[o, 2]) / h - 0.5
            i0, j0 = (int(min(max(math.floor(t) - 1, 0), c - 4)) for t, c in ((tx, X), (ty, Y)))

            def lagrange(t):
                return np.array([np.prod([(t - b) / (a - b) for b in range(4) if b != a]) for a in range(4)])

            prices[o] = lagrange(ty - j0) @ U[q, j0:j0 + 4, i0:i0 + 4] @ lagrange(tx - i0)
            if o == largest:
                lattice = U[q].reshape(-1).copy()
    return prices, lattice


def _coarse_inputs(u, v, axis, mirrored):
    """The 18 inputs of every cell's evaluation across its +axis face (mirrored: the cell across, read back to front)."""
    across = 1 if axis == 2 else 2
    out = []
    for f in (u, v):
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                step = (1 - a) if mirrored else a  # the cell across is one on (the last cell's face is closed)
                n, idx = f.shape[axis], torch.arange(f.shape[axis], device="cuda")
                g = f.index_select(axis, (idx + step).clamp(0, n - 1))
                m, jdx = f.shape[across], torch.arange(f.shape[across], device="cuda")
                out.append(g.index_select(across, (jdx + b).clamp(0, m - 1)))
    return torch.stack(out, -1)


def _coarse_gap(P, u, v, h):
    """The net's correction of both fields (count, n, n), differentiable in the parameters."""
    W1, b1, W2, b2, W3, b3 = P

    def net(x):
        def gelu(z):
            return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))
        return gelu(gelu(x @ W1 + b1) @ W2 + b2) @ W3 + b3

    total = 0.0
    for axis in (2, 1):
        flux = 0.5 * COARSE["scale"] * (net(_coarse_inputs(u, v, axis, False)) - net(_coarse_inputs(u, v, axis, True)))
        n = u.shape[axis]
        flux = flux.narrow(axis, 0, n - 1)
        zero = torch.zeros_like(flux.narrow(axis, 0, 1))
        total = total + torch.cat([zero, flux], axis) - torch.cat([flux, zero], axis)
    return total[..., 0] / h, total[..., 1] / h


def _coarse_parameters(seed):
    flat = torch.tensor(_coarse_net(seed), device="cuda", dtype=torch.float64).requires_grad_(True)
    P, at = [], 0
    for shape in ((18, 64), (64,), (64, 64), (64,), (64, 2), (2,)):
        size = math.prod(shape)
        P.append(flat[at:at + size].reshape(shape))
        at += size
    return flat, P


def _agent_noise(case, q):
    """The planner's hashed normals (agents, samples, horizon, 2): splitmix64's finaliser through Box-Muller."""
    def mix(x):
        x = x ^ (x >> np.uint64(30))
        x = x * np.uint64(0xBF58476D1CE4E5B9)
        x = x ^ (x >> np.uint64(27))
        x = x * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))

    ids = q["ids"].astype(np.uint64)[:, None, None, None]
    k = np.arange(case["samples"], dtype=np.uint64)[None, :, None, None]
    t = np.arange(case["horizon"], dtype=np.uint64)[None, None, :, None]
    d = np.arange(2, dtype=np.uint64)
    with np.errstate(over="ignore"):
        own = mix(ids * np.uint64(0x9E3779B97F4A7C15) + np.uint64(1)) ^ mix(np.array([q["tick"]], np.uint64) * np.uint64(0xD1B54A32D192ED03) + np.uint64(2))
        key = mix(own ^ (k << np.uint64(24)) ^ (t << np.uint64(8)) ^ d)
        other = mix(key ^ np.uint64(0x632BE59BD9B4E019))
    u1, u2 = (((v >> np.uint64(40)).astype(np.float64) + 0.5) / 16777216.0 for v in (key, other))
    return np.sqrt(-2.0 * np.log(u1)) * np.cos(2.0 * np.pi * u2)


def _layers(sizes, flat):
    out, at = [], 0
    for ni, no in zip(sizes[:-1], sizes[1:]):
        out.append((flat[at:at + ni * no].reshape(no, ni), flat[at + ni * no:at + ni * no + no]))
        at += ni * no + no
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "conduction":
        h, dt = _conduction_dt(case)
        f = _uniform(case["nx"] * case["ny"] * case["nz"], seed).double().reshape(case["nz"], case["ny"], case["nx"])
        for _ in range(case["steps"]):
            f = f + dt * _diffuse(f, 0.1, h)
        return [f.reshape(-1)] + ([None] if case["judged"] else [])
    if kind == "black_scholes":
        h = 8.0 / case["nx"]
        dt, sig, r = 0.4 * h * h / (0.2 * 0.2), 0.2, 0.05
        f = _payoff(case["nx"], case["nz"], seed).double().reshape(case["nz"], case["nx"])
        for _ in range(case["steps"]):
            up, dn = _shift(f, 1, 1), _shift(f, 1, -1)
            g = (up - dn) / (2 * h)
            g[:, 0] *= 2
            g[:, -1] *= 2
            f = f + dt * (0.5 * sig * sig * (up - 2 * f + dn) / (h * h) + (r - 0.5 * sig * sig) * g - r * f)
        return [f.reshape(-1)]
    if kind == "implicit":
        shape = (case["nz"], case["ny"], case["nx"])
        h = 1.0 / max(shape)
        f = _uniform(math.prod(shape), 2 * seed).double().reshape(shape)
        w = _uniform(math.prod(shape), 2 * seed + 1, 0.5, 2.0).double().reshape(shape)
        for _ in range(case["steps"]):
            if case["axis"] == "x":
                f = _line_solve(-0.25, 1.5, -0.25, f + 0.25 * (_shift(f, 2, 1) - 2 * f + _shift(f, 2, -1)), 2)
            else:
                a = 0.5 * w
                f = _line_solve(-0.5 * a, 1 + a, -0.5 * a, _line_solve(-a, 1 + 2 * a, -a, f, 1), 0)
        return [f.reshape(-1)]
    if kind == "valley":
        return None  # thresholds and moving heaps: the engine's bits are compared instead
    if kind == "heston":
        return _heston_exact(case, seed)
    if kind == "rollout":
        u, v = (t.double() for t in _coarse_states(case, seed))
        h, dt = 2.0 / case["n"], _coarse_dt(case["n"])
        _, P = _coarse_parameters(seed)
        with torch.no_grad():
            for _ in range(case["steps"]):
                ru, rv = _coarse_rates(u, v, h)
                cu, cv = _coarse_gap(P, u, v, h)
                u, v = u + dt * (ru + cu), v + dt * (rv + cv)
        return u, v
    if kind == "train":
        if case["n"] * case["n"] * case["count"] > 300000:
            return None
        s = _coarse_states(case, seed)
        u, v = (t.double() for t in s)
        h, dt = 2.0 / case["n"], _coarse_dt(case["n"])
        ru, rv = _coarse_rates(u, v, h)
        u1 = (u + dt * (ru + 0.3 * _normal(u.shape, seed + 7).double())).float().double()
        v1 = (v + dt * (rv + 0.3 * _normal(u.shape, seed + 8).double())).float().double()
        flat, P = _coarse_parameters(seed)
        cu, cv = _coarse_gap(P, u, v, h)
        loss = (((cu - ((u1 - u) / dt - ru)) ** 2).sum() + ((cv - ((v1 - v) / dt - rv)) ** 2).sum()) / (2 * u.numel())
        loss.backward()
        return float(loss.detach()), flat.grad.cpu().numpy()
    if kind == "adjoint":
        shape = (case["nz"], case["ny"], case["nx"])
        h, dt = _transport_dt(case)
        start = [_uniform(math.prod(shape), 4 * seed + i, 0.2, 1.0).double().reshape(shape) for i in range(3)]
        D = torch.tensor([0.05, 0.02, 0.01], device="cuda", dtype=torch.float64)

        def step(a, b, c, D):
            def rate(f, k):
                return (_diffuse(f, k, h) - 0.3 * (f - _shift(f, 2, -1)) / h + 0.2 * (_shift(f, 1, 1) - f) / h - 0.1 * (f - _shift(f, 0, -1)) / h)
            m = a * b - 0.1 * c
            return a + dt * (rate(a, D[0]) - m), b + dt * (rate(b, D[1]) - m), c + dt * (rate(c, D[2]) + m)

        states = [start]
        with torch.no_grad():
            for _ in range(case["steps"] - 1):
                states.append(list(step(*states[-1], D)))
        zero = torch.zeros(shape, device="cuda", dtype=torch.float64)
        grads = [zero, zero, _normal((math.prod(shape),), 4 * seed + 3).double().reshape(shape)]
        sums = torch.zeros_like(D)
        for s in reversed(states):
            leaves = [f.detach().requires_grad_(True) for f in s]
            k = D.clone().requires_grad_(True)
            back = torch.autograd.grad(step(*leaves, k), leaves + [k], grad_outputs=grads)
            grads, sums = list(back[:3]), sums + back[3]
        return [g.reshape(-1) for g in grads], [sums[i:i + 1] for i in range(3)]
    if kind == "mppi":
        q = _plan_inputs(case, seed)
        noise = _agent_noise(case, q)
        noise[:, 0] = 0.0
        acts = torch.tensor(np.clip(q["mean"][:, None].astype(np.float64) + 0.3 * noise, -1.0, 1.0), device="cuda")
        net = [tuple(torch.tensor(v, device="cuda", dtype=torch.float64) for v in layer) for layer in _layers(q["sizes"], q["flat"])]
        target = torch.tensor(q["target"], device="cuda", dtype=torch.float64)
        s = torch.tensor(q["obs"], device="cuda", dtype=torch.float64)[:, None].expand(-1, case["samples"], -1)
        cost = torch.zeros(acts.shape[:2], device="cuda", dtype=torch.float64)
        for t in range(case["horizon"]):
            x = torch.cat([s, acts[:, :, t]], -1)
            for k, (W, b) in enumerate(net):
                x = x @ W.T + b
                x = torch.tanh(x) if k < 2 else x
            s = s + 0.1 * x
            cost = cost + ((s - target) ** 2).sum(-1) + 0.01 * (acts[:, :, t] ** 2).sum(-1)
        low = cost.min(1, keepdim=True).values
        lam = torch.clamp(0.25 * (cost.mean(1, keepdim=True) - low), min=1e-4)
        w = torch.exp(-(cost - low) / lam)
        return ((w[:, :, None, None] * acts).sum(1) / w.sum(1)[:, None, None]).cpu().numpy()
    sizes, image, x, t = _learn_inputs(case, seed)
    base = (2 * sizes[0] + 1 + 3) // 4 * 4
    act = {"tanh": torch.tanh, "relu": torch.relu, "silu": torch.nn.functional.silu,
           "gelu": lambda z: torch.nn.functional.gelu(z, approximate="tanh")}[case["act"]]
    head = torch.tensor(image[:base], device="cuda", dtype=torch.float64)
    flat = torch.tensor(image[base:], device="cuda", dtype=torch.float64).requires_grad_(True)
    X = (torch.tensor(x, device="cuda", dtype=torch.float64) - head[:sizes[0]]) * head[sizes[0]:2 * sizes[0]]
    T = torch.tensor(t, device="cuda", dtype=torch.float64)
    m1, m2, losses = torch.zeros_like(flat), torch.zeros_like(flat), []
    for step in range(1, 9):
        y = X
        for k, (W, b) in enumerate(_layers(sizes, flat)):
            y = y @ W.T + b
            y = act(y) if k < 2 else y
        loss = 0.5 * ((y * head[2 * sizes[0]] - T) ** 2).sum() / X.shape[0]
        (g,) = torch.autograd.grad(loss, flat)
        g = g.clamp(-5.0, 5.0)
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        with torch.no_grad():
            flat = (flat - 2e-3 * (m1 / (1 - 0.9 ** step)) / (torch.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)).requires_grad_(True)
        losses.append(float(loss.detach()))
    return losses, np.concatenate([image[:base].astype(np.float64), flat.detach().cpu().numpy()])

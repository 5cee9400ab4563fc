"""The work that a user of this package has it do, as cases that can be timed.

Most cases are whole stretches of a monodomain run: a tissue is set to a given
potential and state (a wave that has crossed part of the domain) and advanced
by a number of time steps, as a program does between two of its outputs.  Two
solve a system on an unstructured mesh, one takes the gradient of a sensor
loss.  The sizes are those of the configurations the package is built for (the
64 x 64 x 16 box, the 400 x 400 x 100 box with and without fibrosis, the batch
of cables and sheets, the 256 x 256 sheet with fitted fields), and smaller and
odd ones of the same kinds.

exact() repeats a case in 64 bits with plain torch operations: the model
equations, the finite-volume rows and the linear solves written out here.
"""
import ctypes
import math

import numpy as np
import torch

import monoalg3d_c_amd as mono
from monoalg3d_c_amd import adjoint, batch

DT = 0.02  # ms, the time step of every configuration
H = 100.0  # um, the cell size
BETA, CM = 0.14, 1.0
REL_TOL = 1e-10  # relative CG residual of every configuration
# a restart inside a beat: the next stimulus is far off
STIM = (1.0e6, 2.0, -50.0, 500.0, 0.0)
MODELS = {"tt2006": mono.MODEL_TT2006, "ord2011": mono.MODEL_ORD2011, "ms2003": mono.MODEL_MS2003}
PRECISIONS = {"fp64": mono.FP64, "fp32": mono.FP32_REFINE}

# a cell at rest (the model's initial state) and 12 ms after it was stimulated
REST = {
    "tt2006": [-85.23, 0.00621, 0.4712, 0.0095, 0.00172, 0.7444, 0.7045, 3.373e-5, 0.7888, 0.9755, 0.9953, 0.999998,
               2.42e-8, 0.000126, 3.64, 0.00036, 0.9073, 8.604, 136.89],
    "ord2011": [-85.0, 7.0, 7.0, 145.0, 145.0, 1e-4, 1e-4, 1.2, 1.2, 0.0, 1.0, 1.0, 1.0, 1.0, 1.0, 0.0, 1.0, 1.0, 0.0,
                1.0, 1.0, 0.0, 1.0, 1.0, 0.0, 1.0, 1.0, 1.0, 1.0, 1.0, 0.0, 1.0, 1.0, 0.0, 0.0, 0.0, 0.0, 1.0, 0.0,
                0.0, 0.0],
    "ms2003": [8.204e-6, 0.8789655],
}
ACTIVE = {
    "tt2006": [18.27, 0.9116, 0.01547, 0.02386, 0.9995, 3.162e-11, 3.122e-11, 0.9708, 0.7402, 0.6422, 0.436, 0.0779,
               0.4742, 0.0004051, 3.164, 1.46, 0.5394, 8.611, 136.9],
    "ord2011": [37.68, 7.003, 7.003, 145.0, 145.0, 0.0001025, 0.0007074, 1.202, 1.072, 0.9999, 9.239e-11, 1.184e-6,
                0.01401, 0.01054, 0.05376, 1.0, 0.9422, 0.9803, 0.9558, 0.0882, 0.6305, 0.9174, 0.1791, 0.7218, 1.0,
                0.2138, 0.9892, 0.2103, 0.8981, 0.8639, 0.7597, 0.5395, 0.536, 0.5661, 0.994, 0.01316, 0.2525, 1.0,
                0.054, 0.06313, 5.134e-5],
    "ms2003": [0.9346, 0.8154],
}
# arithmetic operations of one cell and step of the model, roughly
MODEL_FLOPS = {"tt2006": 900, "ord2011": 2200, "ms2003": 20}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one fibre: the smallest run a user makes, all launches and latency
        tissue("cable 300, TT2006 FP64", "tt2006", (300, 1, 1), "fp64", "isotropic", 50),
        # the first configuration: a small slab, Vm saved every 1 ms (50 steps)
        tissue("box 64x64x16, TT2006 FP64", "tt2006", (64, 64, 16), "fp64", "isotropic", 50),
        # the sheet of a parameter fit, forward only: per-cell conductivities
        tissue("sheet 256x256, MS2003 FP32", "ms2003", (256, 256, 1), "fp32", "factors", 50),
        # a wedge of odd size, isotropic with scars, in the mixed precision
        tissue("wedge 147x101x33, TT2006 FP32, scars", "tt2006", (147, 101, 33), "fp32", "isotropic", 20, 0.1),
        # a patient mesh: a fibre direction of its own in every cell
        tissue("wedge 121x110x37, ORd FP32, own fibres", "ord2011", (121, 110, 37), "fp32", "fibre field", 10),
        # 10% fibrosis in a layered wall, both precisions
        tissue("wall 203x151x40, ORd FP64, fibrosis", "ord2011", (203, 151, 40), "fp64", "layered", 5, 0.1),
        tissue("wall 400x400x50, ORd FP32, fibrosis", "ord2011", (400, 400, 50), "fp32", "layered", 5, 0.1),
        # the headline configuration in both precisions
        tissue("wall 400x400x100, ORd FP64", "ord2011", (400, 400, 100), "fp64", "layered", 5),
        tissue("wall 400x400x100, ORd FP32", "ord2011", (400, 400, 100), "fp32", "layered", 10),
        # the batch configuration: 256 cables and sheets in one run
        {"name": "batch of 256, TT2006 FP32", "kind": "batch", "instances": 256, "cable": 2000, "sheet": 256,
         "precision": "fp32", "steps": 20},
        # the gradient configuration over a shorter stretch (both directions of the adjoint path)
        {"name": "gradient 256x256, 200 steps", "kind": "gradient", "nx": 256, "ny": 256, "steps": 200, "every": 50,
         "checkpoint": 50},
        # an unstructured mesh, matrix and vectors on the device, warm started as every time step is
        {"name": "mesh of 520000 cells, CSR solve", "kind": "mesh", "nx": 130, "ny": 100, "nz": 50, "removed": 0.2,
         "jacobi": False},
    ]


def tissue(name, model, shape, precision, conduction, steps, fibrosis=0.0):
    return {"name": name, "kind": "tissue", "model": model, "nx": shape[0], "ny": shape[1], "nz": shape[2],
            "precision": precision, "conduction": conduction, "steps": steps, "fibrosis": fibrosis}


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["tissue"] * 9 + ["batch", "gradient", "mesh"])
    if kind == "batch":
        return {"kind": kind, "instances": log(8, 256), "cable": log(200, 2000), "sheet": log(40, 256),
                "precision": rng.choice(["fp64", "fp32"]), "steps": 10}
    if kind == "gradient":
        return {"kind": kind, "nx": log(48, 256), "ny": log(48, 256), "steps": rng.choice([60, 100, 150]), "every": 25,
                "checkpoint": rng.choice([0, 50])}
    if kind == "mesh":
        return {"kind": kind, "nx": log(20, 120), "ny": log(20, 100), "nz": log(4, 60),
                "removed": rng.choice([0.1, 0.2, 0.4]), "jacobi": rng.choice([True, False])}
    model = rng.choice(["tt2006", "ord2011", "ord2011", "ms2003"])
    dims = rng.choice([1, 2, 3, 3, 3])
    if dims == 1:
        shape = (log(100, 2000), 1, 1)
    elif dims == 2:
        shape = (log(32, 700), log(32, 700), 1)
    else:
        shape = (log(40, 400), log(40, 400), log(4, 100))
    if dims == 3:
        conduction = rng.choice(["isotropic", "layered", "layered", "fibre field"])
    else:
        conduction = rng.choice(["isotropic", "factors"])
    cells = shape[0] * shape[1] * shape[2]
    if conduction == "fibre field" and cells > 1_000_000:
        conduction = "layered"
    return {"kind": kind, "model": model, "nx": shape[0], "ny": shape[1], "nz": shape[2],
            "precision": rng.choice(["fp64", "fp32"]), "conduction": conduction,
            "steps": 50 if cells < 200_000 else 10 if cells < 2_000_000 else 5,
            "fibrosis": rng.choice([0.0, 0.1]) if dims > 1 and conduction != "factors" else 0.0}


def prepare(case, seed):
    return {"tissue": prepare_tissue, "batch": prepare_batch, "gradient": prepare_gradient,
            "mesh": prepare_mesh}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def exact(case, seed):
    return {"tissue": exact_tissue, "batch": exact_batch, "gradient": exact_gradient,
            "mesh": exact_mesh}[case["kind"]](case, seed)


def work(case):
    """Per time step every state and the potential read and written once, and
    the operations of the model and of one product with the operator."""
    if case["kind"] == "mesh":
        cells = round(case["nx"] * case["ny"] * case["nz"] * (1 - case["removed"]))
        entries = cells * (1 + 6 * (1 - case["removed"]))
        return {"bytes": entries * 12 + cells * (8 + 3 * 8), "flops": 2 * entries}
    if case["kind"] == "gradient":
        cells, model, w, n = case["nx"] * case["ny"], "ms2003", 8, 2
        steps = 2 * case["steps"]
    elif case["kind"] == "batch":
        cells = case["instances"] * (0.5 * (case["cable"] + 100) / 2 + 0.5 * ((case["sheet"] + 32) / 2) ** 2)
        model, steps = "tt2006", case["steps"]
        w, n = (8 if case["precision"] == "fp64" else 4), len(REST[model])
    else:
        cells, model, steps = case["nx"] * case["ny"] * case["nz"], case["model"], case["steps"]
        w, n = (8 if case["precision"] == "fp64" else 4), len(REST[model])
    return {"bytes": steps * cells * (2 * (n - 1) * w + 2 * 8), "flops": steps * cells * (MODEL_FLOPS[model] + 60)}


# ---------------------------------------------------------------------------
# tissues
# ---------------------------------------------------------------------------

class DeviceArray:
    """Memory that a tissue owns, for torch.  Torch keeps this object as long
    as a tensor over the memory lives, and this object keeps the tissue."""

    def __init__(self, owner, pointer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": shape, "typestr": typestr, "version": 2}


def device_views(t, precision):
    """(potential, states) of a tissue as torch tensors over its own buffers."""
    v, sv, pitch, _ = t.device_ptrs()
    typestr = "<f8" if precision == "fp64" else "<f4"
    return (torch.as_tensor(DeviceArray(t, v, (t.n,), "<f8"), device="cuda"),
            torch.as_tensor(DeviceArray(t, sv, (t.neq, pitch), typestr), device="cuda")[:, :t.n])


def generator(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def wave(model, shape, gen, dtype):
    """Potential and states of a wave part of the way through a box: rest ahead
    of a front of random position and direction, a recently activated cell
    behind it, everything modulated by a few per cent over some millimetres."""
    nx, ny, nz = shape
    u = torch.rand(12, generator=gen, device="cuda", dtype=torch.float64).tolist()
    x = torch.arange(nx, device="cuda", dtype=torch.float64).view(1, 1, nx)
    y = torch.arange(ny, device="cuda", dtype=torch.float64).view(1, ny, 1)
    z = torch.arange(nz, device="cuda", dtype=torch.float64).view(nz, 1, 1)
    angle = (u[0] - 0.5) * 0.6 * math.pi
    along = math.cos(angle) * (x - (0.35 + 0.3 * u[1]) * nx) + math.sin(angle) * (y - 0.5 * ny)
    along = along + 4.0 * torch.sin(0.11 * y + 6.28 * u[2]) + 3.0 * torch.sin(0.17 * z + 6.28 * u[3])
    behind = torch.sigmoid(-along / 4.0).reshape(-1)
    waves = [torch.sin((0.05 + 0.06 * u[4 + k]) * x + (0.04 + 0.05 * u[8 + k]) * y + 0.08 * z + 1.7 * k).reshape(-1)
             for k in range(4)]
    rest, active = REST[model], ACTIVE[model]
    states = torch.empty((len(rest), nx * ny * nz), device="cuda", dtype=dtype)
    for k in range(len(rest)):
        states[k] = ((rest[k] + (active[k] - rest[k]) * behind) * (1.0 - 0.01 * (1.0 + waves[k % 4]))).to(dtype)
    v = (rest[0] + (active[0] - rest[0]) * behind) * (1.0 - 0.01 * (1.0 + waves[0]))
    return v, states


def tissue_inputs(case, seed):
    """What a program knows of its tissue: the potential, the states, which
    cells conduct, and the conductivity (keyword arguments of Tissue)."""
    shape = case["nx"], case["ny"], case["nz"]
    gen = generator(seed)
    dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
    v, states = wave(case["model"], shape, gen, dtype)
    n = v.numel()
    kw = {}
    active = None
    if case["fibrosis"]:
        active = torch.rand(n, generator=gen, device="cuda") >= case["fibrosis"]
        active[n // 2] = True
        kw["active"] = active.to(torch.uint8).cpu().numpy()
        v = torch.where(active, v, 0.0)
    if case["conduction"] == "layered":
        kw.update(aniso=True, tensor=layered_tensors(shape[2]), tensor_source=mono.TENSOR_PER_LAYER)
    elif case["conduction"] == "fibre field":
        kw.update(aniso=True, tensor=fibre_field(shape, gen).cpu().numpy(), tensor_source=mono.TENSOR_PER_CELL)
    else:
        kw["tensor"] = mono.iso_tensor(0.00013)
    if case["conduction"] == "factors":
        kw["g_cell"] = torch.exp(0.3 * torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)).cpu().numpy()
    return v, states, active, kw


def layered_tensors(nz):
    """sigma_l / sigma_t = 0.24 / 0.045 S/m, fibres turning from -60 to +60 degrees over the depth."""
    theta = np.deg2rad(-60.0 + 120.0 * np.arange(nz) / max(1, nz - 1))
    return tensors_along(np.cos(theta), np.sin(theta), np.zeros(nz))


def tensors_along(fx, fy, fz):
    lo, dif = 0.000045, 0.00024 - 0.000045
    return np.stack([lo + dif * fx * fx, lo + dif * fy * fy, lo + dif * fz * fz, dif * fx * fy, dif * fx * fz,
                     dif * fy * fz], axis=-1)


def fibre_field(shape, gen):
    """A fibre direction in every cell: the layered one with a smooth disturbance and a transmural part."""
    nx, ny, nz = shape
    u = torch.rand(3, generator=gen, device="cuda", dtype=torch.float64).tolist()
    x = torch.arange(nx, device="cuda", dtype=torch.float64).view(1, 1, nx)
    y = torch.arange(ny, device="cuda", dtype=torch.float64).view(1, ny, 1)
    z = torch.arange(nz, device="cuda", dtype=torch.float64).view(nz, 1, 1)
    theta = math.radians(-60) + math.radians(120) * z / max(1, nz - 1) + 0.3 * torch.sin(0.05 * x + 0.07 * y + 6 * u[0])
    phi = 0.25 * torch.sin(0.06 * x - 0.04 * y + 0.1 * z + 6 * u[1])
    fx, fy, fz = torch.cos(theta) * torch.cos(phi), torch.sin(theta) * torch.cos(phi), torch.sin(phi) + 0 * theta
    lo, dif = 0.000045, 0.00024 - 0.000045
    return torch.stack([lo + dif * fx * fx, lo + dif * fy * fy, lo + dif * fz * fz, dif * fx * fy, dif * fx * fz,
                        dif * fy * fz], dim=-1).reshape(-1, 6)


def prepare_tissue(case, seed):
    v, states, _, kw = tissue_inputs(case, seed)
    t = mono.Tissue((case["nx"], case["ny"], case["nz"]), model=MODELS[case["model"]], dt=DT,
                    precision=PRECISIONS[case["precision"]], cg_tol=0.0, cg_rel_tol=REL_TOL, cg_max_its=500, stim=STIM,
                    **kw)
    return {"run": run_tissue, "tissue": t, "own": device_views(t, case["precision"]), "start": (v, states),
            "steps": case["steps"]}


def run_tissue(s):
    v, states = s["own"]
    v.copy_(s["start"][0])
    states.copy_(s["start"][1])
    s["tissue"].step(s["steps"])
    return {"v": v, "states": states[1:]}


def exact_tissue(case, seed):
    v, states, active, kw = tissue_inputs(case, seed)
    rows = Stencil((case["nx"], case["ny"], case["nz"]), kw, active)
    return exact_steps(case["model"], v, states.double(), active, rows, case["steps"], None)


# ---------------------------------------------------------------------------
# the batch of cables and sheets
# ---------------------------------------------------------------------------

def batch_inputs(case, seed):
    """The instances (their sizes are the case's, their conductance factors the
    seed's), and the potential and states of each, those of one instance behind
    those of the one before."""
    sizes = batch.sweep_instances(case["instances"], 4, cable_cells=(100, case["cable"]),
                                  sheet_side=(32, case["sheet"]))
    factors = np.random.default_rng(seed).uniform(0.5, 1.5, (len(sizes), 3)).astype(np.float32)
    instances = [batch.Instance(i.nx, i.ny, (*map(float, f), 1.0)) for i, f in zip(sizes, factors)]
    gen = generator(seed)
    dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
    parts = [wave("tt2006", (i.nx, i.ny, 1), gen, dtype) for i in instances]
    return instances, torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts], dim=1)


def prepare_batch(case, seed):
    instances, v, states = batch_inputs(case, seed)
    b = batch.Batch(instances, dt=DT, precision=PRECISIONS[case["precision"]], tensor=mono.iso_tensor(0.00013),
                    cg_tol=0.0, cg_rel_tol=REL_TOL, cg_max_its=500, stim=STIM)
    cells = torch.from_numpy(np.concatenate([b.layout.cells(i) for i in range(len(instances))])).cuda()
    own_v, own_states = device_views(b.tissue, case["precision"])
    start_v, start_states = own_v.clone(), own_states.clone()
    start_v[cells] = v
    start_states[:, cells] = states
    return {"run": run_batch, "batch": b, "own": (own_v, own_states), "start": (start_v, start_states), "cells": cells,
            "steps": case["steps"]}


def run_batch(s):
    v, states = s["own"]
    v.copy_(s["start"][0])
    states.copy_(s["start"][1])
    s["batch"].step(s["steps"])
    return {"v": v[s["cells"]], "states": states[1:, s["cells"]]}


def exact_batch(case, seed):
    instances, v, states = batch_inputs(case, seed)
    columns, first = [], 0
    for i in instances:
        columns.append(grid_neighbours((i.nx, i.ny, 1), first))
        first += i.nx * i.ny
    columns = torch.cat(columns, dim=1)
    rows = Rows(columns, torch.full(columns.shape, 0.00013 * H, device="cuda", dtype=torch.float64))
    scale = torch.cat([torch.tensor([i.scale[:3]], device="cuda", dtype=torch.float64).expand(i.nx * i.ny, 3)
                       for i in instances]).T
    return exact_steps("tt2006", v, states.double(), None, rows, case["steps"], scale)


def grid_neighbours(shape, first=0):
    """Cell numbers of the six face neighbours of every cell of a box, -1 where there is none."""
    nx, ny, nz = shape
    cell = first + torch.arange(nx * ny * nz, device="cuda").view(nz, ny, nx)
    out = torch.full((6, nz, ny, nx), -1, device="cuda")
    out[0, :, :, 1:], out[1, :, :, :-1] = cell[:, :, :-1], cell[:, :, 1:]
    out[2, :, 1:], out[3, :, :-1] = cell[:, :-1], cell[:, 1:]
    out[4, 1:], out[5, :-1] = cell[:-1], cell[1:]
    return out.reshape(6, -1)


# ---------------------------------------------------------------------------
# the gradient of a sensor loss
# ---------------------------------------------------------------------------

MS_STIM = (0.0, 2.0, 0.2, 500.0, 0.0)


def gradient_inputs(case, seed):
    n = case["nx"] * case["ny"]
    rng = np.random.default_rng(seed)
    g = np.exp(rng.normal(0.0, 0.3, n))
    s = rng.uniform(0.8, 1.2, n).astype(np.float32).astype(np.float64)
    sensors = np.sort(rng.choice(n, size=min(64, n), replace=False)).astype(np.int64)
    records = case["steps"] // case["every"] + 1
    # recordings of another tissue: an upstroke that passes each sensor at its own time
    arrival = 0.05 * (sensors % case["nx"]) * rng.uniform(0.8, 1.2, len(sensors))
    times = np.arange(records)[:, None] * case["every"] * DT
    return g, s, sensors, 0.95 / (1.0 + np.exp(-(times - arrival) / 0.5))


def prepare_gradient(case, seed):
    g, s, sensors, target = gradient_inputs(case, seed)
    return {"run": run_gradient, "shape": (case["nx"], case["ny"], 1), "g": g, "s": s, "sensors": sensors,
            "target": target, "steps": case["steps"], "every": case["every"], "checkpoint": case["checkpoint"]}


def run_gradient(s):
    loss, dg, ds, traces = adjoint.sensor_loss_grad(s["shape"], s["sensors"], s["steps"], s["every"], s["target"],
                                                    checkpoint_every=s["checkpoint"], g=s["g"], s=s["s"])
    return {"loss": loss, "dg": dg, "ds": ds, "traces": traces}


def exact_gradient(case, seed):
    g, s, sensors, target = (torch.from_numpy(a).cuda() for a in gradient_inputs(case, seed))
    shape = case["nx"], case["ny"], 1
    n = g.numel()
    columns = grid_neighbours(shape)
    there = columns >= 0
    other = torch.where(there, g[columns.clamp(min=0)], 0.0)
    sigma = 0.00013
    face = torch.where(there, 2.0 * sigma * H * g * other / (g + other), 0.0)
    dface = torch.where(there, 2.0 * sigma * H * other * other / (g + other) ** 2, 0.0)
    rows = Rows(columns, face)
    stimulated = (torch.arange(n, device="cuda") % case["nx"] + 0.5) * H < MS_STIM[3]
    v = torch.full((n,), float(np.float32(0.00000820413566106744)), device="cuda", dtype=torch.float64)
    h = torch.full((n,), float(np.float32(0.8789655121804799)), device="cuda", dtype=torch.float64)
    path, time = [(v, h)], 0.0
    for _ in range(case["steps"]):
        stim = torch.where(stimulated, MS_STIM[2] if MS_STIM[0] <= time <= MS_STIM[0] + MS_STIM[1] else 0.0, 0.0)
        dv, (h,) = ms2003([v, h], stim, DT, s)
        v = rows.solve(rows.alpha * (v + dv), v)
        path.append((v, h))
        time += DT
    traces = torch.stack([path[k][0][sensors] for k in range(0, case["steps"] + 1, case["every"])])
    res = 2.0 * (traces - target)
    lam, mu, dg, ds = (torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(4))
    w = torch.zeros_like(lam)
    for k in range(case["steps"], 0, -1):
        if k % case["every"] == 0:
            lam[sensors] += res[k // case["every"]]
        w = rows.solve(lam, w)
        v1, (v, h) = path[k][0], path[k - 1]
        dg -= (dface * (w - w[columns.clamp(min=0)]) * (v1 - v1[columns.clamp(min=0)])).sum(0)
        a = rows.alpha * w
        low = v < 0.13
        close = 150.0 * s
        lam = a * (1.0 + DT * (-1.0 / 6.0 + h * (2.0 * v - 3.0 * v * v) / 0.3))
        ds += mu * torch.where(low, 0.0, DT * h * 150.0 / (close * close))
        mu = a * (DT * (v * v * (1.0 - v)) / 0.3) + mu * torch.where(low, 1.0 - DT / 120.0, 1.0 - DT / close)
    loss = float(((traces - target) ** 2).sum())
    return {"loss": loss, "dg": dg, "ds": ds, "traces": traces}


# ---------------------------------------------------------------------------
# unstructured meshes
# ---------------------------------------------------------------------------

def mesh_inputs(case, seed):
    """Face neighbours and conductances of a box with cells taken out (the same
    ones for every seed) and the rest numbered anew, the start and the
    potential of a time step."""
    shape = case["nx"], case["ny"], case["nz"]
    gen = generator(seed)
    v, _ = wave("tt2006", shape, gen, torch.float64)
    n = v.numel()
    kept = torch.rand(n, generator=generator(4), device="cuda") >= case["removed"]
    kept[0] = True
    number = torch.where(kept, torch.cumsum(kept, 0) - 1, -1)
    columns = grid_neighbours(shape)
    columns = torch.where(columns >= 0, number[columns.clamp(min=0)], -1)[:, kept]
    g = torch.exp(0.3 * torch.randn(n, generator=gen, device="cuda", dtype=torch.float64))[kept]
    other = torch.where(columns >= 0, g[columns.clamp(min=0)], 0.0)
    face = torch.where(columns >= 0, 2.0 * 0.00013 * H * g * other / (g + other), 0.0)
    v = v[kept]
    return Rows(columns, face), v, v + 0.4 * torch.sin(0.3 * torch.arange(v.numel(), device="cuda") / case["nx"])


def prepare_mesh(case, seed):
    rows, x0, vm = mesh_inputs(case, seed)
    n = x0.numel()
    ids = torch.arange(n, device="cuda")
    columns = torch.cat([ids[None], rows.columns])
    values = torch.cat([rows.diagonal[None], -rows.face])
    # entries of a row in column order
    columns = torch.where(columns < 0, n, columns)
    columns, order = columns.sort(dim=0)
    values = values.gather(0, order)
    there = (columns < n).T.reshape(-1)
    row_ptr = torch.zeros(n + 1, device="cuda", dtype=torch.int64)
    row_ptr[1:] = torch.cumsum((columns < n).sum(0), 0)
    b = rows.alpha * vm
    return {"run": run_mesh, "n": n, "row_ptr": row_ptr, "col": columns.T.reshape(-1)[there].to(torch.int32),
            "val": values.T.reshape(-1)[there].contiguous(), "b": b, "x0": x0, "x": torch.empty_like(x0),
            "tol": float((b * b).sum()) * REL_TOL ** 2, "jacobi": int(case["jacobi"])}


def run_mesh(s):
    s["x"].copy_(s["x0"])
    its, err = ctypes.c_int(), ctypes.c_double()
    f = mono.lib().mono_cg_csr_device_noalloc
    p = ctypes.c_void_p
    mono.check(f(s["n"], p(s["row_ptr"].data_ptr()), p(s["col"].data_ptr()), p(s["val"].data_ptr()),
                 p(s["b"].data_ptr()), p(s["x"].data_ptr()), ctypes.c_double(s["tol"]), 500, s["jacobi"],
                 ctypes.byref(its), ctypes.byref(err), None), "mono_cg_csr_device_noalloc")
    return {"x": s["x"], "iterations": its.value}


def exact_mesh(case, seed):
    rows, x0, vm = mesh_inputs(case, seed)
    return {"x": rows.solve(rows.alpha * vm, x0), "iterations": None}


# ---------------------------------------------------------------------------
# 64 bits: operators and linear solves
# ---------------------------------------------------------------------------

ALPHA = ((BETA * CM) / DT) * float(np.float32(1e-8)) * (H * H * H)


class Operator:
    alpha = ALPHA

    def solve(self, b, x):
        """Conjugate gradients, started again until the residual no longer falls."""
        bound = 1e-15 * float(torch.linalg.vector_norm(b))
        last = math.inf
        for _ in range(12):
            r = b - self.times(x)
            size = float(torch.linalg.vector_norm(r))
            if size <= bound or size > 0.5 * last:
                break
            last = size
            p, rr, d = r, size * size, torch.zeros_like(x)
            for _ in range(200):
                q = self.times(p)
                a = rr / float(torch.dot(p, q))
                d = d + a * p
                r = r - a * q
                new = float(torch.dot(r, r))
                if new <= (1e-8 * size) ** 2:
                    break
                p, rr = r + (new / rr) * p, new
            x = x + d
        return x


class Rows(Operator):
    """Cells with face neighbours (columns, -1: none) and face conductances."""

    def __init__(self, columns, face):
        self.columns = columns
        self.face = torch.where(columns >= 0, face, 0.0)
        self.diagonal = self.alpha + self.face.sum(0)
        self.at = columns.clamp(min=0)

    def times(self, x):
        return self.diagonal * x - (self.face * x[self.at]).sum(0)


class Stencil(Operator):
    """Finite-volume rows of a box: conductivity `kw` as given to Tissue, cells
    that conduct in `active` (None: all).  Isotropic faces take the harmonic
    mean of their two cells.  With a full tensor a face's normal part takes the
    mean, and the tangential parts the gradients over the neighbour pairs on
    either side of it that are there, with the mean cross conductivity."""

    def __init__(self, shape, kw, active):
        nx, ny, nz = shape
        self.box = (nz, ny, nx)
        one = torch.ones(self.box, device="cuda", dtype=torch.float64)
        live = one if active is None else active.view(self.box).double()
        self.live = live
        self.padded = torch.nn.functional.pad(live, (1,) * 6)
        self.coef = {(0, 0, 0): self.alpha * live}
        tensor = torch.from_numpy(np.asarray(kw["tensor"])).cuda()
        if "aniso" not in kw:
            g = torch.from_numpy(kw["g_cell"]).cuda().view(self.box) if "g_cell" in kw else one
            sigma = torch.nn.functional.pad(tensor[0] * g * live, (1,) * 6)
            for o in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)):
                a, b = self.at(sigma, (0, 0, 0)), self.at(sigma, o)
                both = (a > 0) & (b > 0)
                self.add(o, torch.where(both, -2.0 * a * b / torch.where(both, a + b, 1.0) * H, 0.0))
            for o, c in list(self.coef.items()):
                if o != (0, 0, 0):
                    self.coef[0, 0, 0] = self.coef[0, 0, 0] - c
            return
        if tensor.shape[0] == nz:
            self.tensor = [torch.nn.functional.pad(tensor[:, k].view(nz, 1, 1), (0, 0, 0, 0, 1, 1)) for k in range(6)]
        else:
            self.tensor = [torch.nn.functional.pad(tensor[:, k].view(self.box), (1,) * 6) for k in range(6)]
        component = {(0, 1): 3, (0, 2): 4, (1, 2): 5}
        for axis in range(3):
            for sign in (1, -1):
                o = self.offset({axis: sign})
                face = self.there(o) * live
                normal = face * (self.of(axis, o) + self.of(axis, (0, 0, 0))) / 2.0 * H
                self.add(o, -normal)
                self.add((0, 0, 0), normal)
                for b in range(3):
                    if b == axis:
                        continue
                    c = 3 - axis - b
                    k = component[min(axis, b), max(axis, b)]
                    pairs = [(self.offset({axis: i * sign, c: j, b: 1}), self.offset({axis: i * sign, c: j, b: -1}))
                             for i in (0, 1) for j in (0, 1, -1)]
                    total, count = 0.0, 0.0
                    for p, q in pairs:
                        both = self.there(p) * self.there(q)
                        total = total + both * (self.of(k, p) + self.of(k, q))
                        count = count + 2.0 * both
                    # the mean is divided by the count a second time, as the reference does
                    some = count.clamp(min=1.0)
                    weight = face * sign * H * total / (some * some)
                    for p, q in pairs:
                        w = weight * self.there(p) * self.there(q)
                        self.add(p, -w)
                        self.add(q, w)
        del self.tensor

    @staticmethod
    def offset(parts):
        return parts.get(0, 0), parts.get(1, 0), parts.get(2, 0)

    def at(self, padded, o):
        """The neighbours' values at offset o of an array padded by one."""
        s = [slice(None) if padded.shape[k] == 1 else slice(1 + o[2 - k], padded.shape[k] - 1 + o[2 - k])
             for k in range(3)]
        return padded[s[0], s[1], s[2]]

    def there(self, o):
        return self.at(self.padded, o)

    def of(self, k, o):
        return self.at(self.tensor[k], o)

    def add(self, o, c):
        self.coef[o] = c + (self.coef[o] if o in self.coef else torch.zeros_like(self.live))

    def times(self, x):
        padded = torch.nn.functional.pad(x.view(self.box), (1,) * 6)
        out = torch.zeros(self.box, device="cuda", dtype=torch.float64)
        for o, c in self.coef.items():
            out.addcmul_(c, self.at(padded, o))
        return out.reshape(-1)


def exact_steps(model, v, states, active, rows, steps, scale):
    """`steps` time steps; a cell that does not conduct is stepped from the potential in its state."""
    states = list(states)
    held = states[0].clone()
    chunk = 1 << 21
    for _ in range(steps):
        inside = v if active is None else torch.where(active, v, held)
        after = torch.empty_like(v)
        for a in range(0, v.numel(), chunk):
            part = slice(a, a + chunk)
            y = [inside[part]] + [s[part] for s in states[1:]]
            if model == "ord2011":
                dv, new = ord2011(y, 0.0, DT)
            elif model == "tt2006":
                dv, new = tt2006(y, 0.0, DT, *(scale[:, part] if scale is not None else (1.0, 1.0, 1.0)))
            else:
                dv, new = ms2003(y, 0.0, DT, 1.0)
            after[part] = y[0] + dv
            for s, x in zip(states[1:], new):
                s[part] = x
        b = rows.alpha * after
        if active is not None:
            b = torch.where(active, b, 0.0)
        v = rows.solve(b, v)
    return {"v": v, "states": torch.stack(states[1:])}


# ---------------------------------------------------------------------------
# 64 bits: the cell models.  Each returns the change of the potential and the
# new states.  A parameter that the reference gives as a 32-bit literal is
# rounded to one.
# ---------------------------------------------------------------------------

def r32(x):
    return float(np.float32(x))


def exp(x):
    return torch.exp(x) if torch.is_tensor(x) else math.exp(x)


def sqrt(x):
    return torch.sqrt(x) if torch.is_tensor(x) else math.sqrt(x)


log, expm1, pow = torch.log, torch.expm1, torch.pow


def cube(x):
    return x * x * x


def rl_toward(inf, x, dt, tau):
    return inf + (x - inf) * exp(-dt / tau)


def rl_from(inf, x, dt, tau):
    return inf - (inf - x) * exp(-dt / tau)


def rl_decay(inf, x, decay):
    return inf - (inf - x) * decay


def ms2003(y, stim, dt, tau_close_scale):
    """Mitchell & Schaeffer 2003."""
    V, h = y
    dV = -(V / 6.0) + (h * (V * V * (1.0 - V))) / 0.3 + stim
    dh = torch.where(V < 0.13, (1.0 - h) / 120.0, -h / (150.0 * tau_close_scale))
    return dt * dV, [h + dt * dh]


def tt2006(y, stim, dt, sKr, sCaL, sKs):
    """ten Tusscher & Panfilov 2006, epicardial."""
    V, Xr1, Xr2, Xs, m, h, j, d, f, f2 = y[0], y[1], y[2], y[3], y[4], y[5], y[6], y[7], y[8], y[9]
    fCass, s, r, Ca_i, Ca_SR, Ca_ss, Rp, Na_i = y[10], y[11], y[12], y[13], y[14], y[15], y[16], y[17]
    K_i, R, Tk, F, Cm, V_c, Ko, Nao = y[18], 8314.472, 310.0, r32(96485.3415), 0.185, 0.016404, 5.4, 140.0
    Cao, P_kna, K_mk, P_NaK, K_mNa, K_pCa, V_rel, k1_prime = 2.0, 0.03, 1.0, 2.724, 40.0, 0.0005, 0.102, 0.15
    max_sr, min_sr, EC, Vmax_up, n_alpha, n_gamma, K_sat, Km_Ca = 2.5, 1.0, 1.5, 0.006375, 2.5, 0.35, 0.1, 1.38
    Km_Nai, K_NaCa, g_to = 87.5, 1000.0, 0.294
    g_Kr = 0.153 * sKr
    g_Ks = 0.098 * sKs
    g_CaL = 3.98e-05 * sCaL
    g_Na, g_pK, g_bca, g_pCa, g_K1, g_bna = 14.838, 0.0146, 0.000592, 0.1238, 5.405, 0.00029
    RT = R * Tk
    EK = (RT / F) * log(Ko / K_i)
    EKs = (RT / F) * log((Ko + (P_kna * Nao)) / (K_i + (P_kna * Na_i)))
    ENa = (RT / F) * log(Nao / Na_i)
    ECa = ((0.5 * R * Tk) / F) * log(Cao / Ca_i)
    VmEK = V - EK
    bK1 = ((3.0 * exp(r32(0.0002) * (VmEK + 100.0))) + exp(r32(0.1) * (VmEK - 10.0))) / (1.0 + exp(-0.5 * VmEK))
    aK1 = r32(0.1) / (1.0 + exp(r32(0.06) * (VmEK - 200.0)))
    xK1 = aK1 / (aK1 + bK1)
    IK1 = g_K1 * xK1 * VmEK
    Ito = g_to * r * s * VmEK
    IKr = g_Kr * Xr1 * Xr2 * VmEK * sqrt(Ko / r32(5.4))
    IKs = g_Ks * (Xs * Xs) * (V - EKs)
    IpK = (g_pK * VmEK) / (1.0 + exp((25.0 - V) / r32(5.98)))
    V15 = V - 15.0
    z = (2.0 * V15 * F) / RT
    near = (V >= r32(15.0 - 1.0e-5)) & (V <= r32(15.0 + 1.0e-5))
    ICaL = g_CaL * d * f * f2 * fCass * torch.where(
        near, 2.0 * F * (0.25 * Ca_ss - Cao),
        ((4.0 * V15 * (F * F)) / RT) * ((0.25 * Ca_ss * exp(z)) - Cao) / expm1(z))
    IbCa = g_bca * (V - ECa)
    IpCa = (g_pCa * Ca_i) / (Ca_i + K_pCa)
    INaK = ((((P_NaK * Ko) / (Ko + K_mk)) * Na_i) / (Na_i + K_mNa)) / (1.0 + (r32(0.1245) * exp((r32(-0.1) \
        * V * F) / RT)) + (r32(0.0353) * exp(((-V) * F) / RT)))
    INa = g_Na * (m * m * m) * h * j * (V - ENa)
    IbNa = g_bna * (V - ENa)
    eg1 = exp(((n_gamma - 1.0) * V * F) / RT)
    INaCa = (K_NaCa * ((exp((n_gamma * V * F) / RT) * (Na_i * Na_i * Na_i) * Cao) - (eg1 * (Nao * Nao * Nao) \
        * Ca_i * n_alpha))) / (((Km_Nai * Km_Nai * Km_Nai) + (Nao * Nao * Nao)) * (Km_Ca + Cao) * (1.0 \
        + (K_sat * eg1)))
    xr1_inf = 1.0 / (1.0 + exp((-26.0 - V) / 7.0))
    tau_xr1 = (450.0 / (1.0 + exp((-45.0 - V) / 10.0))) * (6.0 / (1.0 + exp((V + 30.0) / 11.5)))
    xr2_inf = 1.0 / (1.0 + exp((V + 88.0) / 24.0))
    tau_xr2 = (3.0 / (1.0 + exp((-60.0 - V) / 20.0))) * (r32(1.12) / (1.0 + exp((V - 60.0) / 20.0)))
    xs_inf = 1.0 / (1.0 + exp((-5.0 - V) / 14.0))
    tau_xs = ((1400.0 / sqrt(1.0 + exp((5.0 - V) / 6.0))) * (1.0 / (1.0 + exp((V - 35.0) / 15.0)))) + 80.0
    em = 1.0 + exp((r32(-56.86) - V) / r32(9.03))
    m_inf = 1.0 / (em * em)
    a_m = 1.0 / (1.0 + exp((-60.0 - V) / 5.0))
    b_m = (r32(0.1) / (1.0 + exp((V + 35.0) / 5.0))) + (r32(0.1) / (1.0 + exp((V - 50.0) / 200.0)))
    tau_m = a_m * b_m
    eh = 1.0 + exp((V + r32(71.55)) / r32(7.43))
    h_inf = 1.0 / (eh * eh)
    low = V < -40.0
    a_h = torch.where(low, r32(0.057) * exp((-(V + 80.0)) / r32(6.8)), 0.0)
    b_h = torch.where(low, (r32(2.7) * exp(r32(0.079) * V)) + (310000.0 * exp(r32(0.3485) * V)), r32(0.77) \
        / (r32(0.13) * (1.0 + exp((V + r32(10.66)) / r32(-11.1)))))
    a_j = torch.where(low, (((-25428.0 * exp(r32(0.2444) * V)) - (r32(6.948e-06) * exp(r32(-0.04391) * V))) \
        * (V + r32(37.78))) / (1.0 + exp(r32(0.311) * (V + r32(79.23)))), 0.0)
    b_j = torch.where(low, (r32(0.02424) * exp(r32(-0.01052) * V)) / (1.0 + exp(r32(-0.1378) * (V \
        + r32(40.14)))), (r32(0.6) * exp(r32(0.057) * V)) / (1.0 + exp(r32(-0.1) * (V + 32.0))))
    tau_h = 1.0 / (a_h + b_h)
    j_inf = h_inf
    tau_j = 1.0 / (a_j + b_j)
    d_inf = 1.0 / (1.0 + exp((-8.0 - V) / 7.5))
    a_d = (r32(1.4) / (1.0 + exp((-35.0 - V) / 13.0))) + 0.25
    b_d = r32(1.4) / (1.0 + exp((V + 5.0) / 5.0))
    g_d = 1.0 / (1.0 + exp((50.0 - V) / 20.0))
    tau_d = (a_d * b_d) + g_d
    e30 = exp((V + 30.0) / 10.0)
    v27 = V + 27.0
    f_inf = 1.0 / (1.0 + exp((V + 20.0) / 7.0))
    tau_f = (1102.5 * exp((-(v27 * v27)) / 225.0)) + (200.0 / (1.0 + exp((13.0 - V) / 10.0))) + (180.0 / (1.0 \
        + e30)) + 20.0
    f2_inf = (r32(0.67) / (1.0 + exp((V + 35.0) / 7.0))) + r32(0.33)
    tau_f2 = (562.0 * exp((-(v27 * v27)) / 240.0)) + (31.0 / (1.0 + exp((25.0 - V) / 10.0))) + (80.0 / (1.0 + e30))
    cq = Ca_ss / r32(0.05)
    fCass_inf = (r32(0.6) / (1.0 + cq * cq)) + r32(0.4)
    tau_fCass = (80.0 / (1.0 + cq * cq)) + 2.0
    v45 = V + 45.0
    s_inf = 1.0 / (1.0 + exp((V + 20.0) / 5.0))
    tau_s = (85.0 * exp((-(v45 * v45)) / 320.0)) + (5.0 / (1.0 + exp((V - 20.0) / 5.0))) + 3.0
    v40 = V + 40.0
    r_inf = 1.0 / (1.0 + exp((20.0 - V) / 6.0))
    tau_r = (9.5 * exp((-(v40 * v40)) / 1800.0)) + r32(0.8)
    ecs = EC / Ca_SR
    kcasr = max_sr - ((max_sr - min_sr) / (1.0 + ecs * ecs))
    k1 = k1_prime / kcasr
    k3 = 0.06
    css2 = Ca_ss * Ca_ss
    O = (k1 * css2 * Rp) / (k3 + (k1 * css2))
    Irel = V_rel * O * (Ca_SR - Ca_ss)
    K_up = 0.00025
    Iup = Vmax_up / (1.0 + ((K_up * K_up) / (Ca_i * Ca_i)))
    Ileak = r32(0.00036) * (Ca_SR - Ca_i)
    Ixfer = r32(0.0038) * (Ca_ss - Ca_i)
    k2 = r32(0.045) * kcasr
    k4 = r32(0.005)
    cb = Ca_i + r32(0.001)
    sb = Ca_SR + r32(0.3)
    ssb = Ca_ss + r32(0.00025)
    bufc = 1.0 / (1.0 + ((r32(0.2) * r32(0.001)) / (cb * cb)))
    bufsr = 1.0 / (1.0 + ((10.0 * r32(0.3)) / (sb * sb)))
    bufss = 1.0 / (1.0 + ((r32(0.4) * r32(0.00025)) / (ssb * ssb)))
    V_sr, V_ss = r32(0.001094), r32(5.468e-05)
    dV = -(IK1 + Ito + IKr + IKs + ICaL + INaK + INa + IbNa + INaCa + IbCa + IpK + IpCa + stim)
    dRp = ((-k2) * Ca_ss * Rp) + (k4 * (1.0 - Rp))
    dCai = bufc * (((((Ileak - Iup) * V_sr) / V_c) + Ixfer) - ((((IbCa + IpCa) - (2.0 * INaCa)) * Cm) / (2.0 \
        * V_c * F)))
    dCaSR = bufsr * (Iup - (Irel + Ileak))
    dCass = bufss * (((((-ICaL) * Cm) / (2.0 * V_ss * F)) + ((Irel * V_sr) / V_ss)) - ((Ixfer * V_c) / V_ss))
    dNai = ((-(INa + IbNa + (3.0 * INaK) + (3.0 * INaCa))) / (V_c * F)) * Cm
    dKi = ((-((IK1 + Ito + IKr + IKs + IpK + stim) - (2.0 * INaK))) / (V_c * F)) * Cm
    return dt * dV, [rl_toward(xr1_inf, Xr1, dt, tau_xr1),
                     rl_toward(xr2_inf, Xr2, dt, tau_xr2),
                     rl_toward(xs_inf, Xs, dt, tau_xs),
                     rl_toward(m_inf, m, dt, tau_m),
                     rl_toward(h_inf, h, dt, tau_h),
                     rl_toward(j_inf, j, dt, tau_j),
                     rl_toward(d_inf, d, dt, tau_d),
                     rl_toward(f_inf, f, dt, tau_f),
                     rl_toward(f2_inf, f2, dt, tau_f2),
                     rl_toward(fCass_inf, fCass, dt, tau_fCass),
                     rl_toward(s_inf, s, dt, tau_s),
                     rl_toward(r_inf, r, dt, tau_r),
                     dt * dCai + Ca_i,
                     dt * dCaSR + Ca_SR,
                     dt * dCass + Ca_ss,
                     dt * dRp + Rp,
                     dt * dNai + Na_i,
                     dt * dKi + K_i]


def ord2011(y, stim, dt):
    """O'Hara, Virag, Varro & Rudy 2011, endocardial."""
    v, nai, nass, ki, kss, cai, cass, cansr, cajsr = y[0], y[1], y[2], y[3], y[4], y[5], y[6], y[7], y[8]
    m, hf, hs, j, hsp, jp, mL, hL, hLp, a = y[9], y[10], y[11], y[12], y[13], y[14], y[15], y[16], y[17], y[18]
    iF, iS, ap, iFp, iSp, d, ff, fs, fcaf = y[19], y[20], y[21], y[22], y[23], y[24], y[25], y[26], y[27]
    fcas, jca, nca, ffp, fcafp, xrf, xrs, xs1 = y[28], y[29], y[30], y[31], y[32], y[33], y[34], y[35]
    xs2, xk1, Jrelnp, Jrelp, CaMKt, nao, cao, ko = y[36], y[37], y[38], y[39], y[40], 140.0, 1.8, 5.4
    BSRmax, KmBSR, BSLmax, KmBSL, cmdnmax, kmcmdn, trpnmax = 0.047, 0.00087, 1.124, 0.0087, 0.05, 0.00238, 0.07
    kmtrpn, csqnmax, kmcsqn, aCaMK, bCaMK, CaMKo, KmCaM = 0.0005, 10.0, 0.8, 0.05, 0.00068, 0.05, 0.0015
    KmCaMK, R, Tk, F, L, rad = 0.15, 8314.0, 310.0, 96485.0, 0.01, 0.0011
    vcell = r32(1000.0 * r32(3.14)) * rad * rad * L
    Ageo = r32(2.0 * r32(3.14)) * rad * rad + r32(2.0 * r32(3.14)) * rad * L
    Acap = 2 * Ageo
    vmyo = r32(0.68) * vcell
    vnsr = r32(0.0552) * vcell
    vjsr = r32(0.0048) * vcell
    vss = r32(0.02) * vcell
    RTF = R * Tk / F
    RT = R * Tk
    ENa = RTF * log(nao / nai)
    EK = RTF * log(ko / ki)
    EKs = RTF * log((ko + r32(0.01833) * nao) / (ki + r32(0.01833) * nai))
    CaMKb = CaMKo * (1.0 - CaMKt) / (1.0 + KmCaM / cass)
    CaMKa = CaMKb + CaMKt
    vffrt = v * F * F / RT
    vfrt = v * F / RT
    fCaMK = (1.0 / (1.0 + KmCaMK / CaMKa))
    mss = 1.0 / (1.0 + exp((-(v + r32(39.57))) / r32(9.871)))
    Dm = r32(6.765) * exp((v + r32(11.64)) / r32(34.77)) + r32(8.552) * exp(-(v + r32(77.42)) / r32(5.955))
    Em = exp(-dt * Dm)
    m = rl_decay(mss, m, Em)
    eh = exp((v + r32(82.90)) / r32(6.086))
    hss = 1.0 / (1 + eh)
    Dhf = r32(1.432e-5) * exp(-(v + r32(1.196)) / r32(6.285)) + r32(6.149) * exp((v + r32(0.5096)) / r32(20.27))
    Dhs = r32(0.009794) * exp(-(v + r32(17.95)) / r32(28.05)) + r32(0.3343) * exp((v + r32(5.730)) / r32(56.66))
    Ahf = 0.99
    Ahs = 1.0 - Ahf
    hf = rl_decay(hss, hf, exp(-dt * Dhf))
    hs = rl_decay(hss, hs, exp(-dt * Dhs))
    h = Ahf * hf + Ahs * hs
    jss = hss
    Dj = r32(0.02136) * exp(-(v + r32(100.6)) / r32(8.281)) + r32(0.3052) * exp((v + r32(0.9941)) / r32(38.45))
    rtj = Dj / (r32(2.038) * Dj + 1.0)
    j = rl_decay(jss, j, exp(-dt * rtj))
    hssp = 1.0 / (1.0 + eh * exp((r32(89.1) - r32(82.90)) / r32(6.086)))
    hsp = rl_decay(hssp, hsp, exp(-dt * Dhs / 3.0))
    hp = Ahf * hf + Ahs * hsp
    jp = rl_decay(jss, jp, exp(-dt * rtj / r32(1.46)))
    GNa = 75
    INa = GNa * (v - ENa) * m * m * m * ((1.0 - fCaMK) * h * j + fCaMK * hp * jp)
    mLss = 1.0 / (1.0 + exp((-(v + r32(42.85))) / r32(5.264)))
    mL = rl_decay(mLss, mL, Em)
    ehL = exp((v + r32(87.61)) / r32(7.488))
    hLss = 1.0 / (1.0 + ehL)
    thL = 200.0
    hL = rl_from(hLss, hL, dt, thL)
    hLssp = 1.0 / (1.0 + ehL * exp((r32(93.81) - r32(87.61)) / r32(7.488)))
    thLp = 3.0 * thL
    hLp = rl_from(hLssp, hLp, dt, thLp)
    GNaL = 0.0075
    INaL = GNaL * (v - ENa) * mL * ((1.0 - fCaMK) * hL + fCaMK * hLp)
    ea = exp((-(v - r32(14.34))) / r32(14.82))
    ass = 1.0 / (1.0 + ea)
    Da = 1.0 / (r32(1.2089) * (1.0 + exp(-(v - r32(18.4099)) / r32(29.3814)))) + 3.5 / (1.0 + exp((v + 100.0) \
        / r32(29.3814)))
    Ea = exp(-dt * Da / r32(1.0515))
    a = rl_decay(ass, a, Ea)
    iss = 1.0 / (1.0 + exp((v + r32(43.94)) / r32(5.711)))
    DiF = r32(0.3933) * exp((-(v + 100.0)) / 100.0) + r32(0.08004) * exp((v + 50.0) / r32(16.59))
    DiS = r32(0.001416) * exp((-(v + r32(96.52))) / r32(59.05)) + r32(1.780e-8) * exp((v + r32(114.1)) / r32(8.079))
    rtiF = DiF / (r32(4.562) * DiF + 1.0)
    rtiS = DiS / (r32(23.62) * DiS + 1.0)
    AiF = 1.0 / (1.0 + exp((v - r32(213.6)) / r32(151.2)))
    AiS = 1.0 - AiF
    iF = rl_decay(iss, iF, exp(-dt * rtiF))
    iS = rl_decay(iss, iS, exp(-dt * rtiS))
    ii = AiF * iF + AiS * iS
    assp = 1.0 / (1.0 + ea * exp((r32(24.34) - r32(14.34)) / r32(14.82)))
    ap = rl_decay(assp, ap, Ea)
    dti_develop = r32(1.354) + r32(1.0e-4) / (exp((v - r32(167.4)) / r32(15.89)) + exp(-(v - r32(12.23)) \
        / r32(0.2154)))
    e20 = exp((v + 70.0) / 20.0)
    dti_recover = 1.0 - 0.5 / (1.0 + e20)
    rdti = 1.0 / (dti_develop * dti_recover)
    iFp = rl_decay(iss, iFp, exp(-dt * rtiF * rdti))
    iSp = rl_decay(iss, iSp, exp(-dt * rtiS * rdti))
    ip = AiF * iFp + AiS * iSp
    Gto = 0.02
    Ito = Gto * (v - EK) * ((1.0 - fCaMK) * a * ii + fCaMK * ap * ip)
    dss = 1.0 / (1.0 + exp((-(v + r32(3.940))) / r32(4.230)))
    Dd = exp(r32(-0.05) * (v + 6.0)) + exp(r32(0.09) * (v + 14.0))
    d = rl_decay(dss, d, exp(-dt * (Dd / (r32(0.6) * Dd + 1.0))))
    fss = 1.0 / (1.0 + exp((v + r32(19.58)) / r32(3.696)))
    e10 = exp((v + 20.0) / 10.0)
    Dff = r32(0.0045) * (1.0 / e10) + r32(0.0045) * e10
    Dfs = r32(0.000035) * exp(-(v + 5.0) / 4.0) + r32(0.000035) * exp((v + 5.0) / 6.0)
    rtff = Dff / (7.0 * Dff + 1.0)
    Aff = 0.6
    Afs = 1.0 - Aff
    ff = rl_decay(fss, ff, exp(-dt * rtff))
    fs = rl_decay(fss, fs, exp(-dt * (Dfs / (1000.0 * Dfs + 1.0))))
    f = Aff * ff + Afs * fs
    fcass = fss
    e7 = exp((v - 4.0) / 7.0)
    Dfcaf = r32(0.04) * (1.0 / e7) + r32(0.04) * e7
    Dfcas = r32(0.00012) * exp(-v / 3.0) + r32(0.00012) * exp(v / 7.0)
    rtfcaf = Dfcaf / (7.0 * Dfcaf + 1.0)
    Afcaf = r32(0.3) + r32(0.6) / (1.0 + e10 * exp((-10.0 - 20.0) / 10.0))
    Afcas = 1.0 - Afcaf
    fcaf = rl_decay(fcass, fcaf, exp(-dt * rtfcaf))
    fcas = rl_decay(fcass, fcas, exp(-dt * (Dfcas / (100.0 * Dfcas + 1.0))))
    fca = Afcaf * fcaf + Afcas * fcas
    tjca = 75.0
    jca = rl_from(fcass, jca, dt, tjca)
    ffp = rl_decay(fss, ffp, exp(-dt * rtff / 2.5))
    fp = Aff * ffp + Afs * fs
    fcafp = rl_decay(fcass, fcafp, exp(-dt * rtfcaf / 2.5))
    fcap = Afcaf * fcafp + Afcas * fcas
    Kmn, k2n = 0.002, 1000.0
    km2n = jca * 1.0
    kq = 1.0 + Kmn / cass
    kq2 = kq * kq
    anca = 1.0 / (k2n / km2n + kq2 * kq2)
    nca = anca * k2n / km2n - (anca * k2n / km2n - nca) * exp(-km2n * dt)
    e1 = exp(vfrt)
    e2 = e1 * e1
    PhiCaL = 4.0 * vffrt * (cass * e2 - r32(0.341) * cao) / (e2 - 1.0)
    PhiCaNa = 1.0 * vffrt * (0.75 * nass * e1 - 0.75 * nao) / (e1 - 1.0)
    PhiCaK = 1.0 * vffrt * (0.75 * kss * e1 - 0.75 * ko) / (e1 - 1.0)
    zca, PCa = 2.0, 0.0001
    PCap = r32(1.1) * PCa
    PCaNa = r32(0.00125) * PCa
    PCaK = r32(3.574e-4) * PCa
    PCaNap = r32(0.00125) * PCap
    PCaKp = r32(3.574e-4) * PCap
    gate_np = (f * (1.0 - nca) + jca * fca * nca)
    gate_p = (fp * (1.0 - nca) + jca * fcap * nca)
    ICaL = (1.0 - fCaMK) * PCa * PhiCaL * d * gate_np + fCaMK * PCap * PhiCaL * d * gate_p
    ICaNa = (1.0 - fCaMK) * PCaNa * PhiCaNa * d * gate_np + fCaMK * PCaNap * PhiCaNa * d * gate_p
    ICaK = (1.0 - fCaMK) * PCaK * PhiCaK * d * gate_np + fCaMK * PCaKp * PhiCaK * d * gate_p
    xrss = 1.0 / (1.0 + exp((-(v + r32(8.337))) / r32(6.789)))
    Dxrf = r32(0.3652) * exp((v - r32(31.66)) / r32(3.869)) + r32(4.123e-5) * exp((-(v - r32(47.78))) / r32(20.38))
    Dxrs = r32(0.06629) * exp((v - r32(34.70)) / r32(7.355)) + r32(1.128e-5) * exp((-(v - r32(29.74))) / r32(25.94))
    Axrf = 1.0 / (1.0 + exp((v + r32(54.81)) / r32(38.21)))
    Axrs = 1.0 - Axrf
    xrf = rl_decay(xrss, xrf, exp(-dt * (Dxrf / (r32(12.98) * Dxrf + 1.0))))
    xrs = rl_decay(xrss, xrs, exp(-dt * (Dxrs / (r32(1.865) * Dxrs + 1.0))))
    xr = Axrf * xrf + Axrs * xrs
    rkr = 1.0 / ((1.0 + exp((v + 55.0) / 75.0)) * (1.0 + exp((v - 10.0) / 30.0)))
    GKr = 0.046
    IKr = GKr * sqrt(ko / r32(5.4)) * xr * rkr * (v - EK)
    xs1ss = 1.0 / (1.0 + exp((-(v + r32(11.60))) / r32(8.932)))
    Dxs1 = r32(2.326e-4) * exp((v + r32(48.28)) / r32(17.80)) + r32(0.001292) * exp((-(v + 210.0)) / 230.0)
    xs1 = rl_decay(xs1ss, xs1, exp(-dt * (Dxs1 / (r32(817.3) * Dxs1 + 1.0))))
    xs2ss = xs1ss
    Dxs2 = r32(0.01) * (e20 * exp((-50.0 - 70.0) / 20.0)) + r32(0.0193) * exp((-(v + r32(66.54))) / 31.0)
    xs2 = rl_decay(xs2ss, xs2, exp(-dt * Dxs2))
    KsCa = 1.0 + r32(0.6) / (1.0 + pow(r32(3.8e-5) / cai, r32(1.4)))
    GKs = 0.0034
    IKs = GKs * KsCa * xs1 * xs2 * (v - EKs)
    xk1ss = 1.0 / (1.0 + exp(-(v + r32(2.5538) * ko + r32(144.59)) / (r32(1.5692) * ko + r32(3.8115))))
    Dxk1 = exp((-(v + r32(127.2))) / r32(20.36)) + exp((v + r32(236.8)) / r32(69.33))
    xk1 = rl_decay(xk1ss, xk1, exp(-dt * Dxk1 / r32(122.2)))
    rk1 = 1.0 / (1.0 + exp((v + r32(105.8) - r32(2.6) * ko) / r32(9.493)))
    GK1 = 0.1908
    IK1 = GK1 * sqrt(ko) * rk1 * xk1 * (v - EK)
    kna1, kna2, kna3, kasymm, wna, wca, wnaca, kcaon = 15.0, 5.0, 88.12, 12.5, 6.0e4, 6.0e4, 5.0e3, 1.5e6
    kcaoff, qna, qca = 5.0e3, 0.5224, 0.1670
    hca = exp((qca * v * F) / RT)
    hna = exp((qna * v * F) / RT)
    zna, Gncx = 1.0, 0.0008
    h7 = 1.0 + nao / kna3 * (1.0 + 1.0 / hna)
    h8 = nao / (kna3 * hna * h7)
    h9 = 1.0 / h7
    h10 = kasymm + 1.0 + nao / kna1 * (1.0 + nao / kna2)
    h11 = nao * nao / (h10 * kna1 * kna2)
    h12 = 1.0 / h10
    k1 = h12 * cao * kcaon
    k2 = kcaoff
    k3p = h9 * wca
    k3pp = h8 * wnaca
    k3 = k3p + k3pp
    k5 = kcaoff
    k8 = h8 * h11 * wna
    KmCaAct = 150.0e-6
    INaCa_part = []
    for part, na, ca in ((0.8, nai, cai), (0.2, nass, cass)):
        h1 = 1 + na / kna3 * (1 + hna)
        h2 = (na * hna) / (kna3 * h1)
        h3 = 1.0 / h1
        h4 = 1.0 + na / kna1 * (1 + na / kna2)
        h5 = na * na / (h4 * kna1 * kna2)
        h6 = 1.0 / h4
        k4p = h3 * wca / hca
        k4pp = h2 * wnaca
        k4 = k4p + k4pp
        k6 = h6 * ca * kcaon
        k7 = h5 * h2 * wna
        x1 = k2 * k4 * (k7 + k6) + k5 * k7 * (k2 + k3)
        x2 = k1 * k7 * (k4 + k5) + k4 * k6 * (k1 + k8)
        x3 = k1 * k3 * (k7 + k6) + k8 * k6 * (k2 + k3)
        x4 = k2 * k8 * (k4 + k5) + k3 * k5 * (k1 + k8)
        rxs = 1.0 / (x1 + x2 + x3 + x4)
        E1 = x1 * rxs
        E2 = x2 * rxs
        E3 = x3 * rxs
        E4 = x4 * rxs
        cr = KmCaAct / ca
        allo = 1.0 / (1.0 + cr * cr)
        JncxNa = 3.0 * (E4 * k7 - E1 * k8) + E3 * k4pp - E2 * k3pp
        JncxCa = E2 * k2 - E1 * k1
        INaCa_part.append(r32(part) * Gncx * allo * (zna * JncxNa + zca * JncxCa))
    INaCa_i, INaCa_ss = INaCa_part
    INaCa = INaCa_i + INaCa_ss
    k1p, k1m, k2p, k2m, k3p_, k3m, k4p_, k4m = 949.5, 182.4, 687.2, 39.4, 1899.0, 79300.0, 639.0, 40.0
    Knai0, Knao0, delta = 9.073, 27.78, r32(-0.1550)
    Knai = Knai0 * exp((delta * v * F) / (3.0 * R * Tk))
    Knao = Knao0 * exp(((1.0 - delta) * v * F) / (3.0 * R * Tk))
    Kki, Kko, MgADP, MgATP, Kmgatp, H, eP, Khp = 0.5, 0.3582, 0.05, 9.8, 1.698e-7, 1.0e-7, 4.2, 1.698e-7
    Knap, Kxkur = 224.0, 292.0
    P = eP / (1.0 + H / Khp + nai / Knap + ki / Kxkur)
    nn = 1.0 + nai / Knai
    kk = 1.0 + ki / Kki
    on = 1.0 + nao / Knao
    ok = 1.0 + ko / Kko
    den_i = cube(nn) + kk * kk - 1.0
    den_o = cube(on) + ok * ok - 1.0
    a1 = (k1p * cube(nai / Knai)) / den_i
    b1 = k1m * MgADP
    a2 = k2p
    b2 = (k2m * cube(nao / Knao)) / den_o
    kq_ = ko / Kko
    a3 = (k3p_ * (kq_ * kq_)) / den_o
    b3 = (k3m * P * H) / (1.0 + MgATP / Kmgatp)
    a4 = (k4p_ * MgATP / Kmgatp) / (1.0 + MgATP / Kmgatp)
    kiq = ki / Kki
    b4 = (k4m * (kiq * kiq)) / den_i
    x1 = a4 * a1 * a2 + b2 * b4 * b3 + a2 * b4 * b3 + b3 * a1 * a2
    x2 = b2 * b1 * b4 + a1 * a2 * a3 + a3 * b1 * b4 + a2 * a3 * b4
    x3 = a2 * a3 * a4 + b3 * b2 * b1 + b2 * b1 * a4 + a3 * a4 * b1
    x4 = b4 * b3 * b2 + a3 * a4 * a1 + b2 * a4 * a1 + b3 * b2 * a1
    rxs = 1.0 / (x1 + x2 + x3 + x4)
    E1 = x1 * rxs
    E2 = x2 * rxs
    E3 = x3 * rxs
    E4 = x4 * rxs
    zk = 1.0
    JnakNa = 3.0 * (E1 * a3 - E2 * b3)
    JnakK = 2.0 * (E4 * b1 - E3 * a1)
    Pnak = 30
    INaK = Pnak * (zna * JnakNa + zk * JnakK)
    xkb = 1.0 / (1.0 + exp(-(v - r32(14.48)) / r32(18.34)))
    GKb = 0.003
    IKb = GKb * xkb * (v - EK)
    PNab = 3.75e-10
    ev = e1
    PCab = 2.5e-8
    INab = PNab * vffrt * (nai * ev - nao) / (ev - 1.0)
    ICab = PCab * 4.0 * vffrt * (cai * e2 - r32(0.341) * cao) / (e2 - 1.0)
    GpCa = 0.0005
    IpCa = GpCa * cai / (r32(0.0005) + cai)
    dv = -dt * (INa + INaL + Ito + ICaL + ICaNa + ICaK + IKr + IKs + IK1 + INaCa + INaK + INab + IKb + IpCa \
        + ICab + stim)
    CaMKb = CaMKo * (1.0 - CaMKt) / (1.0 + KmCaM / cass)
    CaMKa = CaMKb + CaMKt
    CaMKt = CaMKt + dt * (aCaMK * CaMKb * (CaMKb + CaMKt) - bCaMK * CaMKt)
    JdiffNa = (nass - nai) / 2.0
    JdiffK = (kss - ki) / 2.0
    Jdiff = (cass - cai) / r32(0.2)
    bt = 4.75
    a_rel = 0.5 * bt
    q = 1.5 / cajsr
    q2 = q * q
    q4 = q2 * q2
    q8 = q4 * q4
    Jrel_inf = a_rel * (-ICaL) / (1.0 + q8)
    tau_rel = bt / (1.0 + r32(0.0123) / cajsr)
    tau_rel = tau_rel.clamp(min=0.005)
    Jrelnp = rl_from(Jrel_inf, Jrelnp, dt, tau_rel)
    btp = 1.25 * bt
    a_relp = 0.5 * btp
    Jrel_infp = a_relp * (-ICaL) / (1.0 + q8)
    tau_relp = btp / (1.0 + r32(0.0123) / cajsr)
    tau_relp = tau_relp.clamp(min=r32(0.005))
    Jrelp = rl_from(Jrel_infp, Jrelp, dt, tau_relp)
    fJ = (1.0 / (1.0 + KmCaMK / CaMKa))
    Jrel = (1.0 - fJ) * Jrelnp + fJ * Jrelp
    Jupnp = r32(0.004375) * cai / (cai + r32(0.00092))
    Jupp = r32(2.75 * r32(0.004375)) * cai / (cai + r32(0.00092) - r32(0.00017))
    Jleak = r32(0.0039375) * cansr / 15.0
    Jup = (1.0 - fJ) * Jupnp + fJ * Jupp - Jleak
    Jtr = (cansr - cajsr) / 100.0
    nai = nai + dt * (-(INa + INaL + 3.0 * INaCa_i + 3.0 * INaK + INab) * Acap / (F * vmyo) + JdiffNa * vss / vmyo)
    nass = nass + dt * (-(ICaNa + 3.0 * INaCa_ss) * Acap / (F * vss) - JdiffNa)
    ki = ki + dt * (-(Ito + IKr + IKs + IK1 + IKb + stim - 2.0 * INaK) * Acap / (F * vmyo) + JdiffK * vss / vmyo)
    kss = kss + dt * (-(ICaK)*Acap / (F * vss) - JdiffK)
    c1 = kmcmdn + cai
    c2 = kmtrpn + cai
    c1s = c1 * c1
    c2s = c2 * c2
    Bcai = (c1s * c2s) / (c1s * c2s + cmdnmax * kmcmdn * c2s + trpnmax * kmtrpn * c1s)
    cai = cai + dt * (Bcai * (-(IpCa + ICab - 2.0 * INaCa_i) * Acap / (2.0 * F * vmyo) - Jup * vnsr / vmyo \
        + Jdiff * vss / vmyo))
    c3 = KmBSR + cass
    c4 = KmBSL + cass
    c3s = c3 * c3
    c4s = c4 * c4
    Bcass = (c3s * c4s) / (c3s * c4s + BSRmax * KmBSR * c4s + BSLmax * KmBSL * c3s)
    cass = cass + dt * (Bcass * (-(ICaL - 2.0 * INaCa_ss) * Acap / (2.0 * F * vss) + Jrel * vjsr / vss - Jdiff))
    cansr = cansr + dt * (Jup - Jtr * vjsr / vnsr)
    c5s = (kmcsqn + cajsr) * (kmcsqn + cajsr)
    Bcajsr = c5s / (c5s + csqnmax * kmcsqn)
    cajsr = cajsr + dt * (Bcajsr * (Jtr - Jrel))
    return dv, [nai, nass, ki, kss, cai, cass, cansr, cajsr, m, hf, hs, j, hsp, jp, mL, hL, hLp, a, iF, iS, ap, iFp,
                iSp, d, ff, fs, fcaf, fcas, jca, nca, ffp, fcafp, xrf, xrs, xs1, xs2, xk1, Jrelnp, Jrelp, CaMKt]

"""What a user of the engine has it do, as cases that can be timed and checked.

Particle runs go through `Solver` and `Batch`: a case advances a loaded flow by
one window of steps and reads out what such a run is made for: sampled fields and
drag, or the cell state that is monitored on the way (occupancy, collision
state and totals, drag). The sort operator, one layer of the field operator in both directions, a
prediction and a training step make up the rest. Sizes are those of
cudadsmc_amd/cases.py, cudadsmc_amd/ensemble.py, bench.py and the reference's
configuration files; `draw` varies them over the ranges in between.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
from pathlib import Path

import numpy as np
import torch

import cudadsmc_amd as dm
from cudadsmc_amd import cases as workloads
from cudadsmc_amd import ensemble, neural
from cudadsmc_amd._capi import check, lib

GOLDEN = Path(__file__).resolve().parent.parent / "tests" / "golden"
BOX = (*ensemble.BOX_MIN, *ensemble.BOX_MAX)
DILATIONS = (1, 2, 4, 8, 1, 2, 4, 8)  # the residual blocks of the default field operator
LR = 1.0e-3


# ------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # smallest run: the sparsest member of the ensembles on its own, read out as a sampling window
        {"name": "sphere_10k", "kind": "sphere", "x": 64, "y": 32, "z": 32, "particles": 10000, "subdiv": 3,
         "U": 1800.0, "n": 3.0e19, "r": 0.02, "sampled": True, "steps": 100},
        # c1: a stretch of the transient, with the cell state, collisions and drag monitored at its end
        {"name": "sphere_100k", "kind": "sphere", "x": 64, "y": 32, "z": 32, "particles": 100000, "subdiv": 3,
         "U": 1500.0, "n": 1.0e20, "r": 0.025, "sampled": False, "steps": 100},
        # c2: a sampling window with its fields and drag
        {"name": "sphere_1m", "kind": "sphere", "x": 128, "y": 64, "z": 64, "particles": 1 << 20, "subdiv": 5,
         "U": 1500.0, "n": 1.0e20, "r": 0.025, "sampled": True, "steps": 100},
        # c3, the benchmark workload: a stretch of the transient, monitored the same way
        {"name": "cone_33m", "kind": "cone", "steps": 100},
        # the reference's own benchmark: REFERENCE mode, Mersenne Twister, one SampleStatistics per 100 steps
        {"name": "reference_557k", "kind": "reference", "config": "config_500k.xml", "mt": True, "steps": 100},
        # 64 uneven instances in one batched step: a sampling window of the data generation
        {"name": "ensemble_64", "kind": "ensemble", "members": 64, "draw": 7, "n_max": 500000, "steps": 100},
        # the sort operator on a c2-sized particle set
        {"name": "sort_1m", "kind": "sort", "keys": 1 << 20, "x": 128, "y": 64, "z": 64},
        # one residual layer of the field operator at the training batch, forward and backward
        {"name": "layer_forward", "kind": "layer_forward", "batch": 8, "z": 32, "y": 32, "x": 64, "cin": 96,
         "cout": 96, "dil": 2},
        {"name": "layer_backward", "kind": "layer_backward", "batch": 8, "z": 32, "y": 32, "x": 64, "cin": 96,
         "cout": 96, "dil": 4},
        # one prediction for a warm start: parameters in, fields out
        {"name": "predict_1", "kind": "predict", "batch": 1, "z": 32, "y": 32, "x": 64, "width": 96, "blocks": 8},
        # one training step of the default operator
        {"name": "train_8", "kind": "train", "batch": 8, "z": 32, "y": 32, "x": 64, "width": 96, "blocks": 8},
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["sphere", "sphere", "sphere", "reference", "ensemble", "sort", "layer_forward",
                       "layer_backward", "predict", "train"])
    if kind == "sphere":
        x = int(_log(rng, 32, 160))
        y, z = (max(16, x // 2 + rng.randint(-3, 3)) for _ in range(2))
        return {"kind": kind, "x": x, "y": y, "z": z,
                "particles": int(_log(rng, 1.0e4, min(4.0e6, 64.0 * x * y * z))), "subdiv": rng.randint(3, 5), "U": rng.uniform(600.0, 3000.0),
                "n": _log(rng, 3.0e19, 1.0e21), "r": rng.uniform(0.015, 0.035), "sampled": rng.random() < 0.5,
                "steps": rng.randint(50, 120)}
    if kind == "reference":
        return {"kind": kind, "config": rng.choice(["config_500k.xml", "config_mln.xml"]), "mt": rng.random() < 0.5,
                "steps": rng.randint(100, 130)}
    if kind == "ensemble":
        return {"kind": kind, "members": rng.randint(4, 64), "draw": rng.randint(0, 1 << 20),
                "n_max": int(_log(rng, 5.0e4, 5.0e5)), "steps": rng.randint(40, 100)}
    if kind == "sort":
        x = int(_log(rng, 32, 256))
        return {"kind": kind, "keys": int(_log(rng, 1.0e4, 3.2e7)), "x": x, "y": max(16, x // 2 + rng.randint(-3, 3)),
                "z": max(16, x // 2 + rng.randint(-3, 3))}
    grid = {"batch": rng.randint(1, 8), "z": rng.randint(20, 32), "y": rng.randint(20, 32), "x": rng.randint(40, 64)}
    if rng.random() < 0.5:  # the simulation grid itself
        grid.update(z=32, y=32, x=64)
    if kind in ("layer_forward", "layer_backward"):
        cin, cout = rng.choice([(32, 96), (96, 96), (96, 96), (64, 64), (128, 128)])
        return {"kind": kind, **grid, "cin": cin, "cout": cout, "dil": rng.choice([1, 2, 4, 8])}
    return {"kind": kind, **grid, "width": rng.choice([32, 64, 96, 96]), "blocks": rng.choice([2, 4, 8])}


# ----------------------------------------------------------- particle runs
@functools.lru_cache(maxsize=None)
def _icosphere(r: float, subdiv: int):
    return dm.icosphere(ensemble.CENTER, r, subdiv)


@functools.lru_cache(maxsize=None)
def _cone():
    return workloads.make_case("c3")


def _develop(sol, s, steps: int) -> None:
    sol.InitSystemState(tuple(s.stream_velocity))
    sol.DoBenchmark(steps, s.dt)
    sol.synchronize()


def _sphere(case: dict, seed: int):
    s = ensemble.settings(ensemble.Case(case["U"], case["n"], 200.0, 300.0, case["r"], case["particles"],
                                        seed % (1 << 31)), dt=6.4e-5 / case["x"])
    s.grid_dim[:] = (case["x"], case["y"], case["z"])
    for a in range(3):
        s.cell_size[a] = (s.bmax[a] - s.bmin[a]) / s.grid_dim[a]
    sol = dm.Solver()
    sol.Init(s)
    sol.SetModel(_icosphere(case["r"], case["subdiv"]),
                 grid=tuple(max(1, math.ceil(2.0 * case["r"] / s.cell_size[a])) for a in range(3)))
    _develop(sol, s, 100)
    if case["sampled"]:
        sol.set_sampling(True)
    return sol, s


def _cone_solver(seed: int):
    s, mesh, cgrid = _cone()
    s = type(s).from_buffer_copy(s)
    s.seed = seed % (1 << 31)
    s.n_streams = int(ensemble.tuned("c3", 0))  # the launch layout of the benchmark
    sol = dm.Solver()
    sol.Init(s)
    tile_cells, scatter_grid = (int(ensemble.tuned("c3", 0, f)) for f in ("tile_cells", "scatter_grid"))
    if tile_cells:
        sol.set_tile_cells(tile_cells)
    if scatter_grid:
        sol.set_scatter_grid(scatter_grid)
    sol.SetModel(mesh, grid=cgrid)
    _develop(sol, s, 100)
    return sol, s


def _reference(case: dict, seed: int):
    s = dm.settings_from_file(str(GOLDEN / case["config"]))
    s.benchmark, s.geometry, s.mt = 1, 1, int(case["mt"])
    s.dt = 0.25e-4
    s.seed = 1 + seed % (1 << 31)
    sol = dm.Solver()
    sol.Init(s)
    sol.SetModel(dm.load_raw(str(GOLDEN / "ares.raw")), grid=(5, 5, 20), move=(0.0, 0.0, -3.0))
    _develop(sol, s, 50)
    return sol, s


def _ensemble(case: dict, seed: int):
    members = ensemble.draw_cases(case["members"], case["draw"], N_range=(1.0e4, case["n_max"]),
                                  seed0=seed % (1 << 30))
    sols = [ensemble.make_solver(m) for m in members]
    batch = dm.Batch(sols)
    batch.run(100)
    batch.set_sampling(True)
    batch.synchronize()
    return batch


# -------------------------------------------------------- field operator
def _gen(seed: int):
    return torch.Generator(device="cuda").manual_seed(seed % (1 << 62))


def _normal(g, *shape, scale: float = 1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _layer(case: dict, seed: int) -> dict:
    g = _gen(seed)
    B, shape = case["batch"], (case["z"], case["y"], case["x"])
    M, cin, cout, bf = B * math.prod(shape), case["cin"], case["cout"], torch.bfloat16
    s = {"case": case, "shape": shape, "M": M,
         "x": _normal(g, M, cin, dtype=bf),
         "w": _normal(g, 27, cout, cin, scale=0.2 * math.sqrt(2.0 / (27 * cin)), dtype=bf),
         "b": _normal(g, cout, scale=0.1)}
    if case["kind"] == "layer_forward":
        # a residual block where the widths agree, the first layer elsewhere
        s["res"] = s["x"] if cin == cout else None
        s["y"], s["h"] = (torch.empty(M, cout, dtype=bf, device="cuda") for _ in range(2))
        return s
    s["h"] = _normal(g, M, cout, dtype=bf).clamp_(min=0)
    s["dy"] = _normal(g, M, cout, scale=1.0e-3, dtype=bf)
    s["dz"] = torch.empty_like(s["dy"])
    s["dx"] = torch.empty(M, cin, dtype=bf, device="cuda")
    s["flip"] = torch.empty(27, cin, cout, dtype=bf, device="cuda")
    s["dw"] = torch.empty(27, cout, cin, device="cuda")
    s["db"] = torch.empty(cout, device="cuda")
    s["part"] = torch.empty((M + 4095) // 4096 * 27 * cout * cin, device="cuda")
    s["bpart"] = torch.empty((M + 511) // 512 * cout, device="cuda")
    return s


def _flow_cases(case: dict, seed: int):
    """Normalised parameters and spheres of `batch` ensemble cases."""
    cases = ensemble.draw_cases(case["batch"], seed % (1 << 62))
    p = neural.normalise_params(*([getattr(c, k) for c in cases] for k in ("U", "n", "T_inf", "T_w", "r")))
    return p, np.array([c.sphere() for c in cases], np.float32)


def _operator(case: dict, seed: int):
    return neural.FieldOperator(shape=(case["z"], case["y"], case["x"]), width=case["width"],
                                dilations=DILATIONS[:case["blocks"]], seed=seed % (1 << 31), max_batch=case["batch"])


def _training_batch(case: dict, op, seed: int):
    """Inputs, smooth targets of the fields' scale with sampling noise, and the mask of the usable cells."""
    g = _gen(seed)
    a0 = op.make_inputs(*_flow_cases(case, seed), BOX)
    f = a0.float()
    near = torch.exp(-4.0 * f[:, 3].clamp(min=0))  # 1 at the sphere, decaying with the distance to it
    target = torch.stack([near * (1 + f[:, 4]), 1 - near, 0.3 * near * f[:, 1], 0.3 * near * f[:, 2],
                          near * (1 + f[:, 8])], 1)
    target = (target + _normal(g, len(f), 5, scale=0.1)).contiguous()
    mask = ((f[:, 3] > 0) & (torch.rand(len(f), generator=g, device="cuda") > 0.05)).float()
    return a0, target, mask


# ----------------------------------------------------------------- prepare
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "sphere":
        sol, s = _sphere(case, seed)
        return {"case": case, "sol": sol, "dt": s.dt}
    if kind == "cone":
        sol, s = _cone_solver(seed)
        return {"case": case, "sol": sol, "dt": s.dt}
    if kind == "reference":
        sol, s = _reference(case, seed)
        return {"case": case, "sol": sol, "dt": s.dt}
    if kind == "ensemble":
        return {"case": case, "batch": _ensemble(case, seed)}
    if kind == "sort":
        # the cells of particles stored in cell order, a tenth of which have moved to a neighbour, a few of them out
        g = _gen(seed)
        n, x, y, cells = case["keys"], case["x"], case["y"], case["x"] * case["y"] * case["z"]
        keys = torch.randint(cells, (n,), generator=g, device="cuda").sort().values
        step = torch.tensor([1, -1, x, -x, x * y, -x * y], device="cuda")
        moved = step[torch.randint(6, (n,), generator=g, device="cuda")]
        u = torch.rand(n, generator=g, device="cuda")
        keys = torch.where(u < 0.1, (keys + moved).clamp(0, cells - 1), keys)
        keys = torch.where(u > 0.999, 0xFFFFFFFF, keys)
        work = torch.empty(int(lib().dsmc_op_sort_work_words(n, cells)), dtype=torch.int32, device="cuda")
        return {"case": case, "keys": keys.to(torch.int32), "cells": cells, "work": work,
                "perm": torch.empty(n, dtype=torch.int32, device="cuda"),
                "start": torch.empty(cells + 1, dtype=torch.int32, device="cuda")}
    if kind in ("layer_forward", "layer_backward"):
        return _layer(case, seed)
    op = _operator(case, seed)
    if kind == "predict":
        params, spheres = _flow_cases(case, seed)
        return {"case": case, "op": op, "params": params, "spheres": spheres}
    a0, target, mask = _training_batch(case, op, seed)
    return {"case": case, "op": op, "a0": a0, "target": target, "mask": mask}


# --------------------------------------------------------------------- run
def _ptr(t) -> C.c_void_p:
    return C.c_void_p(t.data_ptr())


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind in ("sphere", "cone"):
        sol = state["sol"]
        sol.DoBenchmark(case["steps"], state["dt"])
        if case.get("sampled"):
            return {"fields": sol.fields(), "drag": sol.drag()}
        return {"cell_start": sol.cell_start().view(np.int32), "ntc": sol.ntc_state(),
                "collisions": sol.collision_stats(), "drag": sol.drag()}
    if kind == "reference":
        sol = state["sol"]
        sol.DoBenchmark(case["steps"], state["dt"])
        collisions, stats = sol.SampleStatistics()
        return {"collisions": collisions, "stats": stats}
    if kind == "ensemble":
        batch = state["batch"]
        batch.run(case["steps"])
        batch.synchronize()
        fields = [s.fields() for s in batch.solvers]
        return {"fields": {k: np.stack([f[k] for f in fields]) for k in fields[0]},
                "drag": np.stack([s.drag() for s in batch.solvers])}
    if kind == "sort":
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        check(lib().dsmc_op_sort(_ptr(state["keys"]), case["keys"], state["cells"], _ptr(state["perm"]),
                                 _ptr(state["start"]), _ptr(state["work"]), stream))
        return {"perm": state["perm"], "cell_start": state["start"]}
    if kind == "layer_forward":
        s = state
        neural.conv_fwd(s["x"], s["w"], s["b"], case["batch"], s["shape"], case["cin"], case["cout"], 27, case["dil"],
                        relu=True, res=s["res"], y=s["y"], h=s["h"])
        return {"y": s["y"], "h": s["h"]}
    if kind == "layer_backward":
        s, cin, cout = state, case["cin"], case["cout"]
        neural.weight_flip(s["w"], s["flip"], 27, cout, cin)
        neural.relu_bwd(s["dy"], s["h"], s["dz"])
        neural.conv_bwd_w(s["x"], s["dz"], s["dw"], s["part"], case["batch"], s["shape"], cin, cout, 27, case["dil"])
        neural.bias_grad(s["dz"], s["M"], cout, s["db"], s["bpart"])
        neural.conv_fwd(s["dz"], s["flip"], None, case["batch"], s["shape"], cout, cin, 27, case["dil"],
                        res=s["dy"] if cin == cout else None, y=s["dx"])
        return {"dz": s["dz"], "dw": s["dw"], "db": s["db"], "dx": s["dx"]}
    op = state["op"]
    if kind == "predict":
        return op.predict(state["params"], state["spheres"], BOX)
    loss = op.train_step(state["a0"], state["target"], state["mask"], case["batch"], LR)
    M = case["batch"] * case["z"] * case["y"] * case["x"]
    # the weights without the biases: those start at zero, so Adam's first step leaves only their gradients' signs
    return {"loss": loss, "pred": op.pred[:M], "grads": op.grads,
            "weights": {k: v for k, v in op.params.items() if k.startswith("w")}}


# -------------------------------------------------------------------- work
def _conv_work(M: int, cin: int, cout: int, taps: int) -> float:
    return 2.0 * M * taps * cin * cout


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("sphere", "cone", "reference", "ensemble"):
        # per step: positions and velocities read and written, the collision state of each cell read and written,
        # on sampled steps the five sums of each cell too; a move and its collisions are about 100 operations
        if kind == "sphere":
            n, cells, sampled = case["particles"], case["x"] * case["y"] * case["z"], case["sampled"]
        elif kind == "cone":
            n, cells, sampled = 1 << 25, 256 * 128 * 128, False
        elif kind == "reference":
            cells, sampled = 32 ** 3, False
            n = cells * {"config_500k.xml": 17, "config_mln.xml": 32}[case["config"]]
        else:
            members = ensemble.draw_cases(case["members"], case["draw"], N_range=(1.0e4, case["n_max"]))
            n, cells, sampled = sum(m.N for m in members), len(members) * math.prod(ensemble.GRID), True
        return {"bytes": float(case["steps"] * (48 * n + (96 if sampled else 16) * cells)),
                "flops": float(case["steps"] * 100 * n)}
    if kind == "sort":
        n, cells = case["keys"], case["x"] * case["y"] * case["z"]
        return {"bytes": 8.0 * n + 4.0 * (cells + 1), "flops": 0.0}
    M = case["batch"] * case["z"] * case["y"] * case["x"]
    if kind == "layer_forward":
        cin, cout = case["cin"], case["cout"]
        return {"bytes": 2.0 * (M * (cin + 2 * cout) + 27 * cin * cout), "flops": _conv_work(M, cin, cout, 27)}
    if kind == "layer_backward":
        cin, cout = case["cin"], case["cout"]
        return {"bytes": 2.0 * (M * (2 * cin + 3 * cout) + 27 * cin * cout) + 4.0 * (27 * cin * cout + cout),
                "flops": 2 * _conv_work(M, cin, cout, 27)}
    W, L = case["width"], case["blocks"]
    weights = 27 * 32 * W + L * 27 * W * W + 32 * W
    flops = _conv_work(M, 32, W, 27) + L * _conv_work(M, W, W, 27) + _conv_work(M, W, 32, 1)
    if kind == "predict":
        return {"bytes": 20.0 * M + 2.0 * weights, "flops": flops}
    # inputs, targets, mask and prediction; gradients, and weights with both moments in and out
    return {"bytes": (64.0 + 20 + 4 + 128) * M + 28.0 * weights, "flops": 3 * flops - _conv_work(M, 32, W, 27)}


# ------------------------------------------------------------------- exact
def _shifted(x, t: int, taps: int, dil: int):
    """x (B, Z, Y, X, C) read at the offset of tap t, zero outside the grid, as (M, C)."""
    d = [0, 0, 0] if taps == 1 else [(t // 9 - 1) * dil, (t // 3 % 3 - 1) * dil, (t % 3 - 1) * dil]
    out = torch.zeros_like(x)
    to, frm = [slice(None)], [slice(None)]
    for k in range(3):
        n = x.shape[k + 1]
        to.append(slice(max(0, -d[k]), max(0, min(n, n - d[k]))))
        frm.append(slice(max(0, d[k]), max(0, min(n, n + d[k]))))
    if all(abs(d[k]) < x.shape[k + 1] for k in range(3)):
        out[tuple(to)] = x[tuple(frm)]
    return out.reshape(-1, x.shape[-1])


def _conv64(x, w, grid, dil: int):
    v = x.reshape(*grid, x.shape[-1])
    out = torch.zeros(x.shape[0], w.shape[1], dtype=torch.float64, device=x.device)
    for t in range(w.shape[0]):
        out += _shifted(v, t, w.shape[0], dil) @ w[t].T.contiguous()
    return out


def _conv64_grad_x(dy, w, grid, dil: int):
    return _conv64(dy, w.flip(0).transpose(1, 2).contiguous(), grid, dil)


def _conv64_grad_w(x, dy, taps: int, grid, dil: int):
    v, dyt = x.reshape(*grid, x.shape[-1]), dy.T.contiguous()
    return torch.stack([dyt @ _shifted(v, t, taps, dil) for t in range(taps)])


def _inputs64(case: dict, params, spheres):
    """Operator inputs: cell centres in [-1, 1], distance to the sphere in box heights, the case's parameters."""
    B, Z, Y, X = case["batch"], case["z"], case["y"], case["x"]
    f64 = dict(dtype=torch.float64, device="cuda")
    fz, fy, fx = torch.meshgrid(*((torch.arange(n, **f64) + 0.5) / n for n in (Z, Y, X)), indexing="ij")
    lo, hi = torch.tensor(BOX[:3], **f64), torch.tensor(BOX[3:], **f64)
    f = torch.stack([fx, fy, fz], -1)
    out = torch.zeros(B, Z, Y, X, neural.C_IN, **f64)
    out[..., :3] = 2.0 * f - 1.0
    sph = torch.from_numpy(spheres).to(**f64)
    for b in range(B):
        dist = (lo + f * (hi - lo) - sph[b, :3]).square().sum(-1).sqrt() - sph[b, 3]
        out[b, ..., 3] = dist / (hi[1] - lo[1])
        out[b, ..., 4:9] = torch.from_numpy(params[b]).to(**f64)
    return out.reshape(-1, neural.C_IN)


def _net64(case: dict, op, a0) -> dict:
    """Forward pass of the operator's network on FP32 master weights, in 64 bits."""
    grid = (case["batch"], case["z"], case["y"], case["x"])
    p = {k: v.double() for k, v in op.params.items()}
    h = (_conv64(a0, p["w0"], grid, 1) + p["b0"]).clamp(min=0)
    xs, hs = [h], [h]
    for i, d in enumerate(op.dil):
        hs.append((_conv64(xs[-1], p[f"w{i + 1}"], grid, d) + p[f"b{i + 1}"]).clamp(min=0))
        xs.append(xs[-1] + hs[-1])
    return {"p": p, "grid": grid, "xs": xs, "hs": hs, "pred": _conv64(xs[-1], p["wh"], grid, 1) + p["bh"]}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("sphere", "cone", "reference", "ensemble"):
        return None  # FP32 trajectories under random draws: there is no 64-bit value that they approach
    if kind == "sort":
        s = prepare(case, seed)
        keys = s["keys"].long() & 0xFFFFFFFF
        order = keys.clamp(max=s["cells"]).sort(stable=True)
        start = torch.searchsorted(order.values, torch.arange(s["cells"] + 1, device="cuda"))
        return {"perm": order.indices.to(torch.int32), "cell_start": start.to(torch.int32)}
    if kind in ("layer_forward", "layer_backward"):
        s = prepare(case, seed)
        grid, dil = (case["batch"], *s["shape"]), case["dil"]
        x, w = s["x"].double(), s["w"].double()
        if kind == "layer_forward":
            h = (_conv64(x, w, grid, dil) + s["b"].double()).clamp(min=0)
            return {"y": h + x if s["res"] is not None else h, "h": h}
        dz = torch.where(s["h"] > 0, s["dy"].double(), 0.0)
        dx = _conv64_grad_x(dz, w, grid, dil)
        return {"dz": dz, "dw": _conv64_grad_w(x, dz, 27, grid, dil), "db": dz.sum(0),
                "dx": dx + s["dy"].double() if case["cin"] == case["cout"] else dx}
    s = prepare(case, seed)
    op = s["op"]
    if kind == "predict":
        net = _net64(case, op, _inputs64(case, s["params"], s["spheres"]))
        return net["pred"][:, :neural.N_FIELDS].reshape(*net["grid"], neural.N_FIELDS)
    net = _net64(case, op, s["a0"].double())
    mask = s["mask"].double()[:, None]
    diff = (net["pred"][:, :neural.N_FIELDS] - s["target"].double()) * mask
    inv = 1.0 / (float(mask.sum()) * neural.N_FIELDS)
    dpred = torch.zeros_like(net["pred"])
    dpred[:, :neural.N_FIELDS] = 2.0 * diff * inv
    p, grid, xs, hs, L = net["p"], net["grid"], net["xs"], net["hs"], len(op.dil)
    g = {"wh": _conv64_grad_w(xs[L], dpred, 1, grid, 1), "bh": dpred.sum(0)}
    dx = _conv64_grad_x(dpred, p["wh"], grid, 1)
    for i in range(L, 0, -1):
        dz = dx * (hs[i] > 0)
        g[f"w{i}"], g[f"b{i}"] = _conv64_grad_w(xs[i - 1], dz, 27, grid, op.dil[i - 1]), dz.sum(0)
        dx = dx + _conv64_grad_x(dz, p[f"w{i}"], grid, op.dil[i - 1])
    dz = dx * (hs[0] > 0)
    g["w0"], g["b0"] = _conv64_grad_w(s["a0"].double(), dz, 27, grid, 1), dz.sum(0)
    # the first Adam step from zero moments: both bias-corrected moments are the gradient's own
    weights = {k: p[k] - LR * g[k] / (g[k].abs() + 1.0e-8) for k in p if k.startswith("w")}
    return {"loss": (diff * diff).sum() * inv, "pred": net["pred"], "grads": g, "weights": weights}

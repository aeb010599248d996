"""The work that programs have this library do, as timed cases.

A case is one call of a public entry point on data that a program already
holds: a resident grid swept N times with the tuner's launch (api.Grid.run), a
batch of uneven grids (api.Batch.run), or the whole host call of the PSkel API
(api.Stencil2D.runIterativeAutoGPU: upload, sweeps, download).  The sizes are
those of the benchmark's workloads, and odd ones around them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from pskel_amd import api, tuner
from pskel_amd import kernels as K
from pskel_amd.tuner import batch as batch_tuner

DEVICE = "cuda"
SEED16 = 17      # stochastic rounding seed of 16-bit grids
BATCH_LO, BATCH_HI = 64, 2048  # sides of the batched grids

# products and sums of one cell-update
FLOPS = {"jacobi2d": 4, "diffusion9": 17, "life": 10, "cloudsim": 24, "jacobi3d": 6, "box27": 53}
ELEM = {"f32": 4, "u8": 1, "bf16": 2, "f16": 2}


def listed():
    return [
        # the smallest call: a program stepping a little grid (launches and latency are all of it)
        {"name": "jacobi2d small", "call": "grid", "stencil": "jacobi2d", "storage": "f32", "h": 130, "w": 94, "d": 1,
         "iterations": 16, "residual_every": 0},
        # the benchmark's 2D heat sweep
        {"name": "jacobi2d 2048", "call": "grid", "stencil": "jacobi2d", "storage": "f32", "h": 2048, "w": 2048,
         "d": 1, "iterations": 100, "residual_every": 0},
        # an odd mid-sized automaton run to convergence: the residual every 20 sweeps
        {"name": "diffusion9 odd residual", "call": "grid", "stencil": "diffusion9", "storage": "f32", "h": 1021,
         "w": 1531, "d": 1, "iterations": 60, "residual_every": 20},
        # the benchmark's 9-point diffusion/advection automaton
        {"name": "diffusion9 4096", "call": "grid", "stencil": "diffusion9", "storage": "f32", "h": 4096, "w": 4096,
         "d": 1, "iterations": 100, "residual_every": 0},
        # the benchmark's Game of Life board (with its dead ring)
        {"name": "life 8192", "call": "grid", "stencil": "life", "storage": "u8", "h": 8194, "w": 8194, "d": 1,
         "iterations": 100, "residual_every": 0},
        # the reference's cloud simulation: two field arguments read by every cell
        {"name": "cloudsim 4096", "call": "grid", "stencil": "cloudsim", "storage": "f32", "h": 4096, "w": 4096,
         "d": 1, "iterations": 50, "residual_every": 0},
        # the headline: Jacobi-3D with the FP64 residual every 50 sweeps
        {"name": "jacobi3d 512 f32", "call": "grid", "stencil": "jacobi3d", "storage": "f32", "h": 512, "w": 512,
         "d": 512, "iterations": 100, "residual_every": 50},
        # an ordinary odd 3D volume, no residual
        {"name": "jacobi3d odd f32", "call": "grid", "stencil": "jacobi3d", "storage": "f32", "h": 150, "w": 243,
         "d": 211, "iterations": 40, "residual_every": 0},
        # the headline with bf16 storage, stochastic rounding, automatic offset
        {"name": "jacobi3d 512 bf16", "call": "grid", "stencil": "jacobi3d", "storage": "bf16", "h": 512, "w": 512,
         "d": 512, "iterations": 100, "residual_every": 50},
        # a user's own mask, for which there is no specialised kernel: a 3D weighted
        # 3x3x3 box whose faces read the halo value
        {"name": "box27 halo", "call": "grid", "stencil": "box27", "storage": "f32", "h": 192, "w": 225, "d": 260,
         "iterations": 12, "residual_every": 0},
        # many uneven grids advanced together
        {"name": "batch 48", "call": "batch", "count": 48, "shape_seed": 5, "iterations": 105},
        # the PSkel program: host arrays in, host arrays out, everything in between
        {"name": "life host call", "call": "host", "stencil": "life", "storage": "u8", "h": 1000, "w": 1503, "d": 1,
         "iterations": 200, "residual_every": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["jacobi2d", "diffusion9", "life", "cloudsim", "jacobi3d", "jacobi3d", "jacobi3d 16", "box27",
                       "batch", "host"])
    if kind == "batch":
        return {"call": "batch", "count": rng.randint(8, 48), "shape_seed": rng.randrange(1 << 16),
                "iterations": rng.randint(20, 105)}
    if kind == "host":
        stencil = rng.choice(["life", "jacobi2d"])
        return {"call": "host", "stencil": stencil, "storage": "u8" if stencil == "life" else "f32",
                "h": _log_int(rng, 100, 2000), "w": _log_int(rng, 100, 2000), "d": 1,
                "iterations": rng.randint(20, 200), "residual_every": 0}
    case = {"call": "grid", "stencil": kind.split()[0], "storage": "f32", "d": 1}
    if kind in ("jacobi3d", "jacobi3d 16", "box27"):
        lo, hi = (32, 256) if kind == "box27" else (40, 480)
        case.update(h=_log_int(rng, lo, hi), w=_log_int(rng, lo, hi), d=_log_int(rng, lo, hi))
        if kind == "jacobi3d 16":
            case["storage"] = rng.choice(["bf16", "f16"])
        case["iterations"] = rng.randint(6, 12 if kind == "box27" else 100)
    else:
        hi = 8194 if kind == "life" else 4096
        case.update(h=_log_int(rng, 64, hi), w=_log_int(rng, 64, hi))
        if kind == "life":
            case["storage"] = "u8"
        case["iterations"] = rng.randint(10, 50 if kind == "cloudsim" else 100)
    case["residual_every"] = rng.choice([0, 0, rng.randint(5, 50)])
    return case


# ---------------------------------------------------------------------------
# inputs: made on the GPU from the seed, with the workloads' distributions
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _ring(a, value):
    a[0], a[-1] = value, value
    a[:, 0], a[:, -1] = value, value
    return a


def _field(case, seed):
    """The initial state (float32 or uint8, on the GPU)."""
    g, s = _gen(seed), case["stencil"]
    h, w, d = case["h"], case["w"], case["d"]
    if s in ("jacobi3d", "box27"):
        a = torch.rand((h, w, d), generator=g, device=DEVICE)
        if s == "jacobi3d":  # faces held at 1
            _ring(a, 1.0)
            a[:, :, 0], a[:, :, -1] = 1.0, 1.0
        return a
    if s == "life":
        return _ring((torch.rand((h, w), generator=g, device=DEVICE) < 0.3).to(torch.uint8), 0)
    if s == "diffusion9":  # Gaussian blobs over a background
        nb = 32
        u = torch.rand((nb, 3), generator=g, device=DEVICE, dtype=torch.float64)
        sigma = max(4.0, min(h, w) / 100.0)
        y = torch.arange(h, device=DEVICE, dtype=torch.float64)
        x = torch.arange(w, device=DEVICE, dtype=torch.float64)
        gy = torch.exp(-((y[None] - u[:, :1] * h) ** 2) / (2 * sigma * sigma)) * (0.5 + 1.5 * u[:, 2:])
        gx = torch.exp(-((x[None] - u[:, 1:2] * w) ** 2) / (2 * sigma * sigma))
        return (0.1 + gy.t().contiguous() @ gx).to(torch.float32)
    if s == "cloudsim":
        return _ring(15.0 + 10.0 * torch.rand((h, w), generator=g, device=DEVICE), 20.0)
    return _ring(torch.rand((h, w), generator=g, device=DEVICE), 0.0)  # jacobi2d


def _winds(case, seed):
    """wind_x and wind_y of every cell (h, w): a swirl of both signs and some jitter."""
    g = _gen(seed + 7919)
    h, w = case["h"], case["w"]
    jx = torch.rand((h, w), generator=g, device=DEVICE) - 0.5
    jy = torch.rand((h, w), generator=g, device=DEVICE) - 0.5
    x = torch.arange(w, device=DEVICE, dtype=torch.float32)[None]
    y = torch.arange(h, device=DEVICE, dtype=torch.float32)[:, None]
    wx = 0.8 * torch.sin(2 * math.pi * x / w) + 0.2 * jx
    wy = 0.8 * torch.cos(2 * math.pi * y / h) + 0.2 * jy
    return wx, wy


BOX27 = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]


def _box27_weights():
    # 3D binomial smoothing, skewed along h so that no two planes weigh the same
    k = {-1: 0.25, 0: 0.5, 1: 0.25}
    return [k[a] * k[b] * k[c] * (1.0 + 0.1 * a) for a, b, c in BOX27]


BOX9 = [(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1)]


def _diffusion9_weights():
    """The automaton's weights: centre 0.5, edges 0.1, corners 0.025, skewed by a wind of 0.02 along w, -0.01 along h."""
    base = {0: (0.5, 0.0), 1: (0.1, 1.0), 2: (0.025, 0.25)}
    return [base[abs(a) + abs(b)][0] - base[abs(a) + abs(b)][1] * (b * 0.02 - a * 0.01) for a, b in BOX9]


HALO = 0.25  # what a HALO stencil reads outside the volume
DT = 0.01    # cloudsim's time step


def _stencil(name):
    if name == "box27":
        return K.Stencil(K.WEIGHTED_SUM, 3, list(BOX27), weights=_box27_weights(), boundary=K.BOUNDARY_HALO,
                         halo_value=HALO)
    if name == "cloudsim":
        return K.cloudsim(DT)
    return getattr(K, name)()


def _shape(case):
    return (case["h"], case["w"], case["d"]) if case["d"] > 1 else (case["h"], case["w"])


def _batch_shapes(case):
    r = np.random.RandomState(case["shape_seed"])
    a, b = math.log(BATCH_LO), math.log(BATCH_HI)
    return [(int(round(math.exp(a + (b - a) * r.rand()))), int(round(math.exp(a + (b - a) * r.rand()))),
             "jacobi" if i % 2 == 0 else "life") for i in range(case["count"])]


def _batch_case(h, w, kind):
    return {"stencil": "life" if kind == "life" else "jacobi2d", "h": h, "w": w, "d": 1}


class _Device:
    """The grid's current buffer to other GPU code (the CUDA array interface)."""

    def __init__(self, grid, info):
        self.grid = grid  # keeps the memory alive as long as the view
        e = info["elem_bytes"]
        strides = [e]
        for n in ([info["pitch"]] if grid.ndim == 2 else [info["pitch"], info["width"]]):
            strides.insert(0, strides[0] * n)
        self.__cuda_array_interface__ = {
            "shape": grid.shape, "strides": tuple(strides), "data": (info["current"], False), "version": 2,
            "typestr": {"u8": "|u1", "f32": "<f4", "bf16": "<i2", "f16": "<f2"}[grid.storage_name]}


def _view(grid):
    t = torch.as_tensor(_Device(grid, grid.info()), device=DEVICE)
    return t.view(torch.bfloat16) if grid.storage_name == "bf16" else t


def prepare(case, seed):
    if case["call"] == "batch":
        shapes = _batch_shapes(case)
        grids = []
        for i, (h, w, kind) in enumerate(shapes):
            g = api.Grid((h, w), "u8" if kind == "life" else "f32")
            g.upload_pair(_field(_batch_case(h, w, kind), seed * 64 + i).cpu().numpy())
            grids.append(g)
        # the family choices the benchmark measured fastest on such batches
        p = batch_tuner.plan(shapes, case["iterations"], life_depth=7, f32_depth=batch_tuner.MARCH)
        stencils = [batch_tuner.stencil_for(kind) for _, _, kind in shapes]
        return {"call": "batch", "grids": grids, "iterations": case["iterations"],
                "batch": api.Batch(grids, stencils, p["rows"], p["depths"], p["march"])}
    host = _field(case, seed).cpu().numpy()
    stencil = _stencil(case["stencil"])
    if case["call"] == "host":
        inp = api.Array2D(case["w"], case["h"], host.dtype)
        out = api.Array2D(case["w"], case["h"], host.dtype)
        inp.hostArray[...] = host
        out.hostArray[...] = host
        mask = api.Mask2D(len(stencil.offsets))
        for i, (dh, dw) in enumerate(stencil.offsets):
            mask.set(i, dh, dw)
        st = api.Stencil2D(inp, out, mask, api.StencilArgs(stencil.kind, coeff=stencil.coeff))
        return {"call": "host", "stencil": st, "out": out, "iterations": case["iterations"]}
    shape, storage = _shape(case), case["storage"]
    if storage in ("bf16", "f16"):
        grid = api.Grid(shape, storage, store_offset="auto", rounding="stochastic", seed=SEED16)
    else:
        grid = api.Grid(shape, storage)
    grid.upload_pair(host)
    state = {"call": "grid", "grid": grid, "stencil": stencil, "iterations": case["iterations"],
             "residual_every": case["residual_every"],
             "cfg": tuner.choose_config(stencil, shape, storage, case["iterations"])}
    if case["stencil"] == "cloudsim":
        # Args2D host arrays are indexed [y, x] with x = h, y = w
        state["fields"] = [api.Field(f.t().contiguous().cpu().numpy()) for f in _winds(case, seed)]
        for slot, f in enumerate(state["fields"]):
            grid.set_field(slot, f)
    return state


def run(state):
    if state["call"] == "batch":
        state["batch"].run(state["iterations"])
        return [_view(g) for g in state["grids"]]
    if state["call"] == "host":
        state["stencil"].runIterativeAutoGPU(state["iterations"])
        return state["out"].hostArray
    st = state["grid"].run(state["stencil"], state["iterations"], residual_every=state["residual_every"],
                           **state["cfg"])
    u = _view(state["grid"])
    if state["residual_every"]:
        return {"u": u, "residuals": np.array(st["residuals"])}
    return u


def work(case):
    """Bytes: the state read once and written once (and the wind fields read once); flops: the
    products and sums of every cell-update."""
    if case["call"] == "batch":
        byts = flops = 0
        for h, w, kind in _batch_shapes(case):
            byts += 2 * h * w * (1 if kind == "life" else 4)
            flops += h * w * case["iterations"] * FLOPS["life" if kind == "life" else "jacobi2d"]
        return {"bytes": byts, "flops": flops}
    cells = case["h"] * case["w"] * case["d"]
    fields = 8 * cells if case["stencil"] == "cloudsim" else 0
    return {"bytes": 2 * cells * ELEM[case["storage"]] + fields,
            "flops": cells * case["iterations"] * FLOPS[case["stencil"]]}


# ---------------------------------------------------------------------------
# the same runs in 64 bits
# ---------------------------------------------------------------------------
def _sweep64(name, u, extra):
    """One sweep of a float64 (life: uint8) state; the ring or faces keep their values."""
    v = u.clone()
    if name == "life":
        n = torch.zeros_like(u[1:-1, 1:-1])
        for a in (0, 1, 2):
            for b in (0, 1, 2):
                if (a, b) != (1, 1):
                    n += u[a:u.shape[0] - 2 + a, b:u.shape[1] - 2 + b]
        v[1:-1, 1:-1] = (n == 3) | ((n == 2) & (u[1:-1, 1:-1] == 1))
    elif name == "jacobi2d":
        v[1:-1, 1:-1] = 0.25 * (u[:-2, 1:-1] + u[2:, 1:-1] + u[1:-1, :-2] + u[1:-1, 2:])
    elif name == "diffusion9":
        acc = torch.zeros_like(u[1:-1, 1:-1])
        for wt, (dh, dw) in zip(extra, BOX9):
            acc += wt * u[1 + dh:u.shape[0] - 1 + dh, 1 + dw:u.shape[1] - 1 + dw]
        v[1:-1, 1:-1] = acc
    elif name == "cloudsim":
        wx, wy = extra
        c, n, s = u[1:-1, 1:-1], u[:-2, 1:-1], u[2:, 1:-1]
        e, w = u[1:-1, 2:], u[1:-1, :-2]
        xw, yw = wx[1:-1, 1:-1], wy[1:-1, 1:-1]
        tx, ty = torch.where(xw > 0, e, w), torch.where(yw > 0, s, n)
        wind = -xw.abs() * ((c - tx) * 10.0) - yw.abs() * ((c - ty) * 10.0)
        v[1:-1, 1:-1] = c + (-0.0243 * ((4.0 * c - (n + e + w + s)) * 0.25)) * DT + wind * DT
    elif name == "jacobi3d":
        i = slice(1, -1)
        v[i, i, i] = extra * (u[:-2, i, i] + u[2:, i, i] + u[i, :-2, i] + u[i, 2:, i] + u[i, i, :-2] + u[i, i, 2:])
    else:  # box27, every cell, HALO outside
        p = torch.nn.functional.pad(u, (1, 1, 1, 1, 1, 1), value=HALO)
        v.zero_()
        for wt, (a, b, c) in zip(extra, BOX27):
            v += wt * p[1 + a:p.shape[0] - 1 + a, 1 + b:p.shape[1] - 1 + b, 1 + c:p.shape[2] - 1 + c]
    return v


def _run64(case, seed, iterations, every=0):
    name = case["stencil"]
    u = _field(case, seed)
    if name != "life":
        u = u.double()
    f32 = lambda x: float(np.float32(x))  # noqa: E731 (the descriptor holds float32 coefficients)
    extra = {"diffusion9": lambda: [f32(x) for x in _diffusion9_weights()],
             "box27": lambda: [f32(x) for x in _box27_weights()],
             "jacobi3d": lambda: f32(1.0 / 6.0),
             "cloudsim": lambda: [x.double() for x in _winds(case, seed)]}.get(name, lambda: None)()
    res = []
    for k in range(1, iterations + 1):
        v = _sweep64(name, u, extra)
        if every and k % every == 0:
            res.append(float((v.double() - u.double()).norm()))
        u = v
    return u, np.array(res)


def exact(case, seed):
    if case["call"] == "batch":
        return [_run64(_batch_case(h, w, kind), seed * 64 + i, case["iterations"])[0]
                for i, (h, w, kind) in enumerate(_batch_shapes(case))]
    u, res = _run64(case, seed, case["iterations"], case["residual_every"])
    if case["call"] == "host":
        return u.cpu().numpy()
    if case["storage"] in ("bf16", "f16"):
        # storage holds u - offset; the offset is the mean of the initial state
        u = u - float(np.float32(_field(case, seed).double().mean().item()))
    return {"u": u, "residuals": res} if case["residual_every"] else u

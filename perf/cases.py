"""The work that users of this library have it do, as cases that can be timed.

A pass advances a lattice (or a batch of lattices) that the program holds by
some time steps through the public entry points and hands back the whole
lattice: the host copy that KernelData.Pdfs points to after Kernel() or a
batch sync.  The geometries, kernels, storage types, sizes and step counts
are those of bench.py, the tests and the driver: channels, pipes, block
arrays and porous media from a few thousand to 16.8 million cells, FP64 and
the shifted FP32 / FP16 storage types, single calls from 20 to 1000 steps,
steady-state solves with their convergence checks, and batches.

The seed sets what differs from run to run of one geometry: the initial
density ramp (KernelSetInitialDensity, src/Kernel.c:288), the viscosity
(omega) and the body force.
"""
import ctypes as C
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "lbm-benchmark-kernels_amd"))
import lbm_amd as lbm  # noqa: E402

MAGIC = 0.1875                                # TRT Lambda 3/16, as bench.py
BYTES = {"fp64": 8, "fp32s": 4, "fp16s": 2}   # of one stored value
TYPES = {"fp64": np.float64, "fp32s": np.float32, "fp16s": np.float16}
F16_SCALE = 4096.0                            # -fp16-scale default
MAX_CELL_STEPS = 256 ** 3 * 300               # of any case
MAX_CALL_STEPS = 1000                         # of one Kernel() call


def listed():
    return [
        # one short call on a very small sample: launch latency decides
        {"name": "list-porous-24-fp64", "kind": "run", "kernel": "list-aa-pv-soa", "geometry": "porous-3-0.7-7",
         "x": 24, "y": 24, "z": 24, "prec": "fp64", "steps": 20},
        # a small full-array channel, as a test or a parameter scan runs it
        {"name": "aa-channel-32-fp32s", "kind": "run", "kernel": "aa-soa", "geometry": "channel",
         "x": 32, "y": 32, "z": 32, "prec": "fp32s", "steps": 100},
        # the small configuration the reference also runs on its CPU
        {"name": "aa-channel-64-fp64", "kind": "run", "kernel": "aa-soa", "geometry": "channel",
         "x": 64, "y": 64, "z": 64, "prec": "fp64", "steps": 1000},
        # a ragged block array through the list kernel
        {"name": "list-blocks-97x61x45-fp64", "kind": "run", "kernel": "list-aa-pv-soa", "geometry": "blocks-6",
         "x": 97, "y": 61, "z": 45, "prec": "fp64", "steps": 300},
        # a permeability solve: chunks of 100 steps, each with its momentum check
        {"name": "steady-porous-96-fp32s", "kind": "steady", "kernel": "list-aa-pv-soa", "geometry": "porous-5-0.75-11",
         "x": 96, "y": 96, "z": 96, "prec": "fp32s", "steps": 600},
        # a ragged pipe in the narrowest storage
        {"name": "aa-pipe-129x83x110-fp16s", "kind": "run", "kernel": "aa-soa", "geometry": "pipe",
         "x": 129, "y": 83, "z": 110, "prec": "fp16s", "steps": 400},
        # a ragged porous sample just above the last-level cache
        {"name": "list-porous-163x150x141-fp32s", "kind": "run", "kernel": "list-aa-pv-soa",
         "geometry": "porous-6-0.8-42", "x": 163, "y": 150, "z": 141, "prec": "fp32s", "steps": 200},
        # many small samples stepped together, one check interval
        {"name": "batch-porous-32x32..96-fp32s", "kind": "batch", "kernel": "list-aa-pv-soa", "samples": 32,
         "sample_seed": 2024, "low": 32, "high": 96, "prec": "fp32s", "steps": 100},
        # a large ragged porous sample in FP16
        {"name": "list-porous-231x200x187-fp16s", "kind": "run", "kernel": "list-aa-pv-soa",
         "geometry": "porous-6-0.8-42", "x": 231, "y": 200, "z": 187, "prec": "fp16s", "steps": 200},
        # the headline workload of bench.py
        {"name": "list-porous-256-fp64", "kind": "run", "kernel": "list-aa-pv-soa", "geometry": "porous-6-0.8-42",
         "x": 256, "y": 256, "z": 256, "prec": "fp64", "steps": 300},
        # the large full-array channel of bench.py, in FP64 and in FP32
        {"name": "aa-channel-256-fp64", "kind": "run", "kernel": "aa-soa", "geometry": "channel",
         "x": 256, "y": 256, "z": 256, "prec": "fp64", "steps": 200},
        {"name": "aa-channel-256-fp32s", "kind": "run", "kernel": "aa-soa", "geometry": "channel",
         "x": 256, "y": 256, "z": 256, "prec": "fp32s", "steps": 200},
    ]


def _edge(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: edges and step counts spread over
    their logarithm, every kernel, storage type and geometry."""
    kind = rng.choice(["run", "run", "run", "steady", "batch"])
    prec = rng.choice(["fp64", "fp64", "fp32s", "fp16s"])
    if kind == "batch":
        low = _edge(rng, 20, 48)
        return {"kind": "batch", "kernel": "list-aa-pv-soa", "samples": rng.randint(8, 48),
                "sample_seed": rng.randrange(1 << 30), "low": low, "high": low + rng.randint(8, 64), "prec": prec,
                "steps": 100}
    kernel = rng.choice(["list-aa-pv-soa", "list-aa-pv-soa", "aa-soa"])
    size = math.exp(rng.uniform(math.log(20), math.log(224)))
    x, y, z = (max(16, min(240, int(round(size * rng.uniform(0.75, 1.3))))) for _ in range(3))
    geometry = rng.choice(["channel", "pipe", "blocks-%d" % rng.randint(2, 8)] if kernel == "aa-soa" else
                          ["channel", "blocks-%d" % rng.randint(2, 8)] +
                          2 * ["porous-%g-%g-%d" % (round(rng.uniform(2.5, 8.0), 2), round(rng.uniform(0.5, 0.9), 3),
                                                    rng.randrange(1, 1 << 30))])
    steps = min(MAX_CALL_STEPS, _edge(rng, 20, 1000), MAX_CELL_STEPS // (2 * x * y * z))
    if kind == "steady":
        steps = max(200, steps // 100 * 100)
    return {"kind": kind, "kernel": kernel, "geometry": geometry, "x": x, "y": y, "z": z, "prec": prec,
            "steps": max(20, steps)}


def _geometry(geometry, dims):
    # x periodic, y and z walls, as bench.py builds every geometry
    return lbm.Geometry.from_string(geometry, dims, (1, 0, 0))


def _samples(case):
    """(dims, geometry) of a batch's samples (the recipe of workloads.py)."""
    rng = random.Random(case["sample_seed"])
    return [(tuple(_edge(rng, case["low"], case["high"]) for _ in range(3)),
             "porous-%.3f-%.4f-%d" % (rng.uniform(3.0, 8.0), rng.uniform(0.5, 0.9), rng.randint(1, 2 ** 31 - 1)))
            for _ in range(case["samples"])]


def _physics(seed, count=1):
    """Per lattice (omega, force, density at the inlet, density at the outlet)."""
    rng = random.Random(seed * 7919 + 17)
    return [(rng.uniform(0.8, 1.6), rng.uniform(0.5e-5, 2e-5), rng.uniform(1.0, 1.02), rng.uniform(0.98, 1.0))
            for _ in range(count)]


def _host_copy(owner, kd, prec, count):
    """The `count` values of the lattice's host copy (KernelData.Pdfs[0]: FP64
    values, or FP32 / FP16 deviations from the weights), in an array that
    keeps `owner`, and with it the memory, alive."""
    t = np.dtype(TYPES[prec])
    buf = (C.c_char * (count * t.itemsize)).from_address(C.cast(kd.contents.Pdfs[0], C.c_void_p).value)
    buf.owner = owner
    return np.frombuffer(buf, t)


def _list_view(owner, kd, prec):
    """[19][nFluid] view of a list lattice's host copy, nodes in list order."""
    info = lbm.LbmHipListInfo()
    lbm.hip_lib().LbmHipListGetInfo(kd, C.byref(info))
    return _host_copy(owner, kd, prec, 19 * info.nCells).reshape(19, info.nCells)[:, :info.nFluid]


def _aa_view(owner, kd, dims, prec):
    """[19][X][Y][Z] view of a full-array lattice's host copy: one ghost layer
    in x and y, z rows padded to whole 128-byte lines, behind one line with
    the z ghost cell in FP16 (walls on both z faces)."""
    X, Y, Z = dims
    line = 128 // BYTES[prec]
    off = line if prec == "fp16s" else 0
    row = -(-(off + Z + (1 if off else 0)) // line) * line
    values = _host_copy(owner, kd, prec, 19 * (X + 2) * (Y + 2) * row)
    return values.reshape(19, X + 2, Y + 2, row)[:, 1:-1, 1:-1, off:off + Z]


def prepare(case, seed):
    """The lattice(s) built and initialised, as a program holds them before it
    steps them."""
    args = ["-lambda", repr(MAGIC), "-prec", case["prec"], "-quiet"]
    if case["kind"] == "batch":
        samples = _samples(case)
        batch = lbm.Batch(args)
        ids = [batch.add(_geometry(g, dims), omega, force)
               for (dims, g), (omega, force, _, _) in zip(samples, _physics(seed, len(samples)))]
        return {"case": case, "batch": batch, "ids": ids}
    dims = (case["x"], case["y"], case["z"])
    geo = _geometry(case["geometry"], dims)
    omega, force, rho_in, rho_out = _physics(seed)[0]
    k = lbm.Kernel(case["kernel"], geo, args)
    # rest state under a density ramp: f = w rho (the initialiser's omega is 1)
    init = lbm.case_data(omega=1.0, rho_in=rho_in, rho_out=rho_out)
    lbm.host_lib().KernelSetInitialDensity(C.byref(geo.ld), k.kd, C.byref(init))
    view = (_aa_view(k, k.kd, dims, case["prec"]) if case["kernel"] == "aa-soa" else
            _list_view(k, k.kd, case["prec"]))
    cd = lbm.case_data(omega=omega, xforce=force, iterations=case["steps"])
    return {"case": case, "kernel": k, "cd": cd, "view": view}


def run(state):
    """The steps of one call and the lattice after them."""
    case = state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        b.sync()
        return [_list_view(b, b.kernel_data(i), case["prec"]) for i in state["ids"]]
    k = state["kernel"]
    if case["kind"] == "steady":
        r = k.run_steady(state["cd"], 100, 0.0, case["steps"])
        return {"lattice": state["view"], "mass": float(r.mass), "momentum": float(r.momentumX)}
    k.run(state["cd"])
    return state["view"]


def work(case):
    """Every fluid node's 19 values read and written once per time step, and
    about 200 operations of the collision (the accounting of the reference's
    MFLUP/s rooflines, doc/main.rst:347, without its adjacency)."""
    if case["kind"] == "batch":
        nodes = sum(_geometry(g, dims).n_fluid for dims, g in _samples(case))
    else:
        nodes = _geometry(case["geometry"], (case["x"], case["y"], case["z"])).n_fluid
    updates = nodes * case["steps"]
    return {"bytes": 2 * 19 * BYTES[case["prec"]] * updates, "flops": 200 * updates}


# ------------------------------------------------- the same steps in 64 bits
_NAMES = "N S E W NE SE NW SW T TN TE TW TS B BS BN BW BE C".split()
_C = [tuple(n.count(p) - n.count(m) for p, m in ("EW", "NS", "TB")) if n != "C" else (0, 0, 0) for n in _NAMES]
_W = [{0: 1 / 3, 1: 1 / 18, 2: 1 / 36}[abs(a) + abs(b) + abs(c)] for a, b, c in _C]
_INV = [_C.index((-a, -b, -c)) for a, b, c in _C]


def _steps64(solid, f, omega, force, steps):
    """TRT collide-stream steps with half-way bounce-back on full arrays
    ([19][X][Y][Z], z fastest) and the body force after every step."""
    even, odd = omega, 1.0 / (0.5 + MAGIC / (1.0 / omega - 0.5))
    dev = f.device
    c = torch.tensor(_C, dtype=torch.float64, device=dev)
    from_solid = [torch.roll(solid, _C[d], (0, 1, 2)) for d in range(19)]
    for _ in range(steps):
        rho = f.sum(0)
        u = torch.tensordot(c.T.contiguous(), f.reshape(19, -1), 1).reshape(3, *rho.shape)
        base = rho - 1.5 * (u * u).sum(0)
        post = torch.empty_like(f)
        for d in range(19):
            i = _INV[d]
            if i < d:
                continue
            cu = _C[d][0] * u[0] + _C[d][1] * u[1] + _C[d][2] * u[2]
            e = even * (0.5 * (f[d] + f[i]) - _W[d] * (base + 4.5 * cu * cu))
            o = odd * (0.5 * (f[d] - f[i]) - _W[d] * 3.0 * cu)
            post[d] = f[d] - e - o
            if i != d:
                post[i] = f[i] - e + o
        for d in range(19):
            f[d] = torch.where(from_solid[d], post[_INV[d]], torch.roll(post[d], _C[d], (0, 1, 2)))
            if _C[d][0]:
                f[d] += 3.0 * _W[d] * _C[d][0] * force
    return f


def _exact_lattice(dims, geometry, physics, ramp, steps):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    omega, force, rho_in, rho_out = physics
    solid = torch.from_numpy(_geometry(geometry, dims).mask.transpose(2, 1, 0) == 0).to(dev)
    rho = torch.ones(dims[0], dtype=torch.float64, device=dev)
    if ramp:
        rho = rho_in + (rho_out - rho_in) * torch.arange(dims[0], dtype=torch.float64, device=dev) / (dims[0] - 1.0)
    f = torch.empty((19, *dims), dtype=torch.float64, device=dev)
    for d in range(19):
        f[d] = _W[d] * rho[:, None, None]
    f = _steps64(solid, f, omega, force, steps + (steps & 1))
    return solid, f


def _stored(solid, f, prec, keep_solid):
    """The lattice as it is stored: f, or the (scaled) deviation from the
    weights; solid cells keep f = 0 in the full array and are left out of the
    list."""
    w = torch.tensor(_W, dtype=torch.float64, device=f.device)
    f[:, solid] = 0.0
    if prec != "fp64":
        f -= w[:, None, None, None]
    if prec == "fp16s":
        f *= F16_SCALE
    return (f if keep_solid else f[:, ~solid]).cpu().numpy()


def exact(case, seed):
    if case["kind"] == "batch":
        samples = _samples(case)
        return [_stored(*_exact_lattice(dims, g, p, False, case["steps"]), case["prec"], False)
                for (dims, g), p in zip(samples, _physics(seed, len(samples)))]
    dims = (case["x"], case["y"], case["z"])
    solid, f = _exact_lattice(dims, case["geometry"], _physics(seed)[0], True, case["steps"])
    aa = case["kernel"] == "aa-soa"
    if case["kind"] == "steady":
        fluid = f[:, ~solid]
        mass = float(fluid.sum())
        momentum = float(sum(_C[d][0] * fluid[d].sum() for d in range(19)))
        return {"lattice": _stored(solid, f, case["prec"], aa), "mass": mass, "momentum": momentum}
    return _stored(solid, f, case["prec"], aa)

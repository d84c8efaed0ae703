"""The work that programs built on this framework have it do, as timed cases.

Each case goes through the public entry points of bhgpu (the ctypes binding
of include/bh_gpu.h) as a user's program calls them:

  step      one force evaluation with kick and drift on particles in device
            memory (bh_step_device, as a graph replay or eagerly), the call an
            integrator makes once per time step
  leapfrog  a whole short run: upload, resident steps, download
  host      one drop-in step_particles call on host records (bh_step)
  batch     one step of many independent systems in one call (bh_step_batch)
  accel     tree build and accelerations with their list lengths
            (bh_build_tree, bh_accel)
  direct    the FP64 direct sum on a subset (bh_direct_sum), the accuracy
            reference of every run
  energy    kinetic and potential energy (bh_energies), the conservation
            check of every run
  serve     independent leapfrog requests through the continuous-batching
            server (bh_server_*)

Inputs are Plummer and Hernquist spheres (G = M = a = 1) and uniform cubes
with velocities, made on the GPU from the seed alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amt-bh-benchmark_amd"))

from bhgpu import autotune, layout  # noqa: E402
from bhgpu import lib as bl  # noqa: E402

DT = 1e-3


def _step(name, ic, n, theta, eps, leaf, target, quad=True, fp64=False, graph=False):
    return {"name": name, "kind": "step", "ic": ic, "n": n, "theta": theta, "eps": eps, "leaf": leaf, "group": 256,
            "target": target, "quad": quad, "fp64": fp64, "graph": graph}


def listed():
    return [
        # the smallest earnest system, called eagerly: latency and launches
        _step("step-1000", "plummer", 1000, 0.5, 1e-2, 16, 32),
        # the small-system latency workload, as a graph replay
        _step("step-4096-graph", "plummer", 4096, 0.5, 1e-2, 16, 32, graph=True),
        # the double-precision accuracy workload's step
        _step("step-65536-fp64", "plummer", 65536, 0.5, 1e-2, 16, 32, fp64=True),
        # monopoles only, at the widest opening angle, a ragged size
        _step("step-100003-monopole", "hernquist", 100003, 0.7, 1e-2, 8, 32, quad=False),
        # the uniform cube (reference driver's leaf capacity)
        _step("step-1M-uniform", "uniform", 1 << 20, 0.6, 1e-3, 8, 32),
        # the headline system
        _step("step-16M-plummer", "plummer", 1 << 24, 0.5, 1e-3, 32, 96),
        # a short resident run with its transfers, odd size
        {"name": "leapfrog-250007", "kind": "leapfrog", "ic": "plummer", "n": 250007, "steps": 10, "theta": 0.5,
         "eps": 1e-2, "leaf": 32, "group": 256, "target": 64, "graph": False},
        # the mixed ensemble: 64 systems, log-uniform sizes, three angles
        {"name": "batch-64-mixed", "kind": "batch", "systems": 64, "n_min": 4096, "n_max": 1 << 20},
        # a force evaluation with lists, as accuracy studies make it
        {"name": "accel-131072-fp64", "kind": "accel", "ic": "hernquist", "n": 131072, "theta": 0.4, "eps": 1e-2,
         "leaf": 16, "group": 256, "target": 32, "fp64": True},
        # the accuracy reference: 4,096 targets of a 1M system
        {"name": "direct-4096-of-1M", "kind": "direct", "ic": "plummer", "n": 1 << 20, "targets": 4096, "eps": 1e-3},
        # the energy check of a medium run
        {"name": "energy-131072", "kind": "energy", "ic": "plummer", "n": 131072},
        # a burst of requests, sizes log-uniform from 1,024
        {"name": "serve-16", "kind": "serve", "requests": 16, "n_min": 1024, "n_max": 131072, "steps_max": 6},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "leapfrog", "host", "batch", "accel", "direct", "energy",
                       "serve"])
    ic = rng.choice(["plummer", "hernquist", "uniform"])
    theta = rng.choice([0.4, 0.5, 0.6, 0.7])
    eps = rng.choice([0.0, 1e-3, 1e-2, 1e-2])
    leaf = rng.choice([8, 16, 32])
    target = rng.choice([32, 64, 96])
    if kind == "step":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 500, 4 << 20), "theta": theta, "eps": eps, "leaf": leaf,
                "group": 256, "target": target, "quad": rng.random() < 0.8, "fp64": rng.random() < 0.25,
                "graph": rng.random() < 0.4}
    if kind == "leapfrog":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 4000, 500000), "steps": rng.randint(4, 12), "theta": theta,
                "eps": 1e-2, "leaf": leaf, "group": 256, "target": target, "graph": rng.random() < 0.4}
    if kind == "host":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 1000, 500000), "theta": theta, "eps": eps, "leaf": leaf,
                "group": 256, "target": target, "quad": True, "fp64": rng.random() < 0.25}
    if kind == "batch":
        return {"kind": kind, "systems": rng.randint(8, 64), "n_min": _log_int(rng, 500, 4096),
                "n_max": _log_int(rng, 8192, 1 << 19)}
    if kind == "accel":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 2000, 200000), "theta": theta, "eps": eps, "leaf": leaf,
                "group": 256, "target": target, "fp64": True}
    if kind == "direct":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 20000, 1 << 20), "targets": _log_int(rng, 256, 4096),
                "eps": eps}
    if kind == "energy":
        return {"kind": kind, "ic": ic, "n": _log_int(rng, 5000, 131072)}
    return {"kind": "serve", "requests": rng.randint(4, 16), "n_min": 1024, "n_max": _log_int(rng, 8192, 131072),
            "steps_max": rng.randint(2, 6)}


# ---- inputs

def _iso(g, n):
    u = torch.rand(2, n, generator=g, device="cuda", dtype=torch.float64)
    c = 2.0 * u[0] - 1.0
    s = torch.sqrt(torch.clamp(1.0 - c * c, min=0.0))
    return torch.stack([s * torch.cos(2.0 * math.pi * u[1]), s * torch.sin(2.0 * math.pi * u[1]), c], dim=1)


def _speed_fraction(g, n):
    """v / v_escape with density q^2 (1 - q^2)^3.5, by a tabulated inverse."""
    q = np.linspace(0.0, 1.0, 4097)
    cdf = np.cumsum(q * q * (1.0 - q * q) ** 3.5)
    cdf = torch.as_tensor(cdf / cdf[-1], device="cuda")
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    return torch.clamp(torch.searchsorted(cdf, u).to(torch.float64) / 4096.0, max=1.0)


def _particles(ic, n, seed):
    """(n, 8) float64 device records with bh_particle's layout: id and pad
    (32 bits each), mass, position, velocity."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    p = torch.zeros(n, 8, device="cuda", dtype=torch.float64)
    p.view(torch.int32)[:, 0] = torch.arange(n, device="cuda", dtype=torch.int32)
    p[:, 1] = 1.0 / n
    if ic == "uniform":
        p[:, 2:5] = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)
        p[:, 5:8] = 2.0 * torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64) - 1.0
        return p
    u = 1.0 - torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    if ic == "plummer":  # r < 10 a
        r = 1.0 / torch.sqrt(torch.pow(u * (1.0 + 1e-2) ** -1.5, -2.0 / 3.0) - 1.0)
        v_esc = math.sqrt(2.0) * torch.pow(1.0 + r * r, -0.25)
    else:  # Hernquist, r < 20 a
        s = torch.sqrt(u) * (20.0 / 21.0)
        r = s / (1.0 - s)
        v_esc = torch.sqrt(2.0 / (1.0 + r))
    p[:, 2:5] = _iso(g, n) * r[:, None]
    p[:, 5:8] = _iso(g, n) * (_speed_fraction(g, n) * v_esc)[:, None]
    return p


def _host(p):
    return p.cpu().numpy().view(layout.PARTICLE).reshape(-1)


def _fields(p):
    """The records' fields, as views."""
    return {"id": p.view(torch.int32)[:, 0], "mass": p[:, 1], "pos": p[:, 2:5], "vel": p[:, 5:8]}


def _host_fields(a):
    return {"id": a["id"].view(np.int32), "mass": a["mass"], "pos": a["pos"], "vel": a["vel"]}


def _fp(c):
    return layout.force_params(c["theta"], c["eps"] ** 2, 1.0, c.get("quad", True))


def _context(c):
    ctx = bl.Context(0)
    if c.get("fp64"):
        ctx.set_precision(bl.BH_FP64)
    if c.get("graph"):
        ctx.set_graph_mode(bl.BH_GRAPH_ON)
    return ctx


def _sizes(c):
    """The case's system sizes: spread over the logarithm of its range, each
    with an offset of its own, so that they are odd and uneven."""
    count = c["systems"] if c["kind"] == "batch" else c["requests"]
    u = [(k + (0.618034 * (k + 1)) % 1.0) / count for k in range(count)]
    return [int(round(c["n_min"] * (c["n_max"] / c["n_min"]) ** f)) for f in u]


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("step", "leapfrog", "host", "accel", "direct", "energy"):
        p = _particles(c["ic"], c["n"], seed)
    if kind == "step":
        return {"c": c, "ctx": _context(c), "fp": _fp(c), "in": p, "out": torch.empty_like(p)}
    if kind in ("leapfrog", "host", "accel"):
        return {"c": c, "ctx": _context(c), "fp": _fp(c), "p": _host(p)}
    if kind == "direct":
        idx = np.sort(np.random.default_rng(seed).choice(c["n"], size=c["targets"], replace=False)).astype(np.uint32)
        return {"c": c, "ctx": _context(c), "p": _host(p), "idx": idx}
    if kind == "energy":
        return {"c": c, "ctx": _context(c), "p": _host(p)}
    if kind == "batch":
        # alternating kinds, three angles, each system with its tuned shapes
        rows, parts = [], []
        for k, n in enumerate(_sizes(c)):
            theta = (0.4, 0.5, 0.7)[k % 3]
            leaf, group, target, tile = autotune.shapes_for(n, theta)
            rows.append(layout.system(n, layout.force_params(theta, 1e-4, 1.0, True), leaf, group, target, DT, DT,
                                      walk_tile=tile))
            parts.append(_particles("plummer" if k % 2 == 0 else "hernquist", n, seed * 1000 + k))
        p = torch.cat(parts)
        return {"c": c, "ctx": _context(c), "systems": np.concatenate(rows), "in": p, "out": torch.empty_like(p)}
    ctx = _context(c)
    work = []
    for k, n in enumerate(_sizes(c)):
        leaf, group, target, _ = autotune.shapes_for(n, 0.5)
        req = bl.request(n, theta=0.5, eps2=1e-4, max_leaf=leaf, group_size=group, target_size=target,
                         steps=1 + 5 * k % c["steps_max"], dt=DT)
        work.append((_host(_particles("plummer", n, seed * 1000 + k)), req))
    return {"c": c, "ctx": ctx, "server": bl.Server(ctx), "work": work}


# ---- one pass

def run(s):
    c, ctx, kind = s["c"], s["ctx"], s["c"]["kind"]
    if kind == "step":
        ctx.step_device(s["in"].data_ptr(), s["out"].data_ptr(), c["n"], s["fp"], c["leaf"], c["group"], c["target"],
                        DT, DT)
        return _fields(s["out"])
    if kind == "leapfrog":
        ctx.state_upload(s["p"])
        for k in range(c["steps"] + 1):
            ctx.state_step(s["fp"], c["leaf"], c["group"], c["target"], DT if 0 < k < c["steps"] else DT / 2,
                           DT if k < c["steps"] else 0.0)
        return _host_fields(ctx.state_download())
    if kind == "host":
        return _host_fields(ctx.step(s["p"], s["fp"], c["leaf"], c["group"], c["target"], DT, DT)[0])
    if kind == "batch":
        ctx.step_batch_device(s["in"].data_ptr(), s["out"].data_ptr(), s["systems"])
        return _fields(s["out"])
    if kind == "accel":
        ctx.build_tree(s["p"], c["leaf"], c["group"])
        acc, n_pp, n_pc, _ = ctx.accel(s["fp"], c["target"])
        return {"acc": acc, "n_pp": n_pp.view(np.int32), "n_pc": n_pc.view(np.int32)}
    if kind == "direct":
        return {"acc": ctx.direct_sum(s["p"], s["idx"], c["eps"] ** 2)}
    if kind == "energy":
        kinetic, potential = ctx.energies(s["p"])
        return {"kinetic": kinetic, "potential": potential}
    server = s["server"]
    order = [server.submit(p, req) for p, req in s["work"]]
    got = {}
    while server.pending() != (0, 0):
        server.step()
        for ticket, result, _ in server.poll():
            got[ticket] = result
    return [_host_fields(got[t]) for t in order]


# ---- what a pass cannot do without

def _tree_flops(n, theta, leaf, target, quad):
    """Interactions of one evaluation, at 19 flops per particle and 55 per
    quadrupole cell. Per particle about 160 (0.5 / theta)^3 (log2(n / leaf) -
    5) cells and the particles of some 44 leaves at theta 0.5 (fitted to
    the lists of Plummer spheres, within a factor of two elsewhere); never
    more than all pairs."""
    f = (0.5 / theta) ** 3
    pc = max(0.0, 160.0 * f * (math.log2(max(n, 2) / leaf) - 5.0))
    pp = min(float(n), 44.0 * f ** 0.5 * max(leaf * 0.6, target * 0.3))
    return n * (19.0 * pp + (55.0 if quad else 19.0) * min(pc, float(n)))


def work(case):
    c, kind = case, case["kind"]
    if kind in ("step", "host"):
        return {"bytes": 128 * c["n"], "flops": _tree_flops(c["n"], c["theta"], c["leaf"], c["target"], c["quad"])}
    if kind == "leapfrog":
        return {"bytes": 128 * c["n"],
                "flops": (c["steps"] + 1) * _tree_flops(c["n"], c["theta"], c["leaf"], c["target"], True)}
    if kind == "accel":
        return {"bytes": (64 + 32) * c["n"], "flops": _tree_flops(c["n"], c["theta"], c["leaf"], c["target"], True)}
    if kind == "direct":
        return {"bytes": 64 * c["n"] + 28 * c["targets"], "flops": 19.0 * c["n"] * c["targets"]}
    if kind == "energy":
        return {"bytes": 64 * c["n"], "flops": 9.0 * c["n"] * c["n"] / 2}
    ns = _sizes(c)
    turns = 1.0 if kind == "batch" else (c["steps_max"] + 1) / 2 + 1
    return {"bytes": 128 * sum(ns), "flops": turns * sum(_tree_flops(n, 0.5, 16, 64, True) for n in ns)}


# ---- the same in 64 bits, by direct summation in torch

EXACT_MAX = 140000


def _direct(pos, mass, targets, eps2, skip):
    """Accelerations of pos[targets]; `skip`: each target's own index."""
    out = torch.empty(len(targets), 3, device="cuda", dtype=torch.float64)
    chunk = max(1, (1 << 25) // len(pos))
    for a in range(0, len(targets), chunk):
        t = targets[a:a + chunk]
        d = [pos[None, :, k] - pos[t][:, k, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + eps2
        w = mass[None, :] / (r2 * torch.sqrt(r2))
        w[torch.arange(len(t), device="cuda"), skip[a:a + chunk]] = 0.0
        for k in range(3):
            out[a:a + chunk, k] = (w * d[k]).sum(dim=1)
    return out


def _morton_order(pos):
    """Ascending 63-bit Morton key of the cell in the padded cube, ties by index."""
    lo, hi = pos.min(dim=0).values, pos.max(dim=0).values
    half = 0.5 * float((hi - lo).max())
    half = (half if half > 0.0 else 1.0) * (1.0 + 1e-9)
    scale = 2097152.0 / (2.0 * half)
    key = torch.zeros(len(pos), device="cuda", dtype=torch.int64)
    for a in range(3):
        corner = 0.5 * (float(lo[a]) + float(hi[a])) - half
        cell = torch.clamp(torch.floor((pos[:, a] - corner) * scale), 0.0, 2097151.0).to(torch.int64)
        for b in range(21):
            key |= ((cell >> b) & 1) << (3 * b + a)
    return torch.sort(key, stable=True).indices


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("leapfrog", "batch", "serve") or (kind != "direct" and c["n"] > EXACT_MAX):
        return None
    p = _particles(c["ic"], c["n"], seed)
    pos, mass, vel = p[:, 2:5].contiguous(), p[:, 1].contiguous(), p[:, 5:8].contiguous()
    every = torch.arange(c["n"], device="cuda")
    if kind == "direct":
        idx = np.sort(np.random.default_rng(seed).choice(c["n"], size=c["targets"], replace=False))
        t = torch.as_tensor(idx.astype(np.int64), device="cuda")
        return {"acc": _direct(pos, mass, t, c["eps"] ** 2, t)}
    if kind == "energy":
        total = 0.0
        chunk = max(1, (1 << 25) // c["n"])
        for a in range(0, c["n"], chunk):
            t = every[a:a + chunk]
            d = pos[None, a:, :] - pos[t][:, None, :]
            r = torch.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2])
            w = mass[t][:, None] * mass[None, a:] / r
            later = every[None, a:] > t[:, None]
            total += float(torch.where(later, w, torch.zeros_like(w)).sum())
        kinetic = float((0.5 * mass * (vel * vel).sum(dim=1)).sum())
        return {"kinetic": kinetic, "potential": -total}
    order = _morton_order(pos)
    acc = _direct(pos, mass, order, c["eps"] ** 2, order)
    if kind == "accel":
        return {"acc": acc, "n_pp": None, "n_pc": None}
    vel = vel[order] + DT * acc
    return {"id": None, "mass": mass[order], "pos": pos[order] + DT * vel, "vel": vel}

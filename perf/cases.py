"""The work this framework is used for, as cases that can be measured.

`listed()` names the cases, `draw(rng)` gives more of the same ranges,
`prepare(case, seed)` makes what a program holds before the call (bodies on
the GPU, a context), `run(state)` is one pass through the public entry points
of `fmms_amd`, `work(case)` counts the bytes and operations a pass cannot do
without, and `exact(case, seed)` gives the same outputs from the FP64 direct
sum.

A case is a dict of plain values:
  entry    accel        tree build and evaluation, device arrays
           accel_host   the same from host arrays (the reference's interface)
           evaluate     evaluation on a tree built beforehand
           leapfrog     `steps` kick-drift-kick steps on device state
           direct       FP64 direct sum at `targets` sampled bodies, host arrays
  model    plummer, hernquist, disk, halos (64 halos in a unit cube), ensemble
           (`systems` Plummer spheres and disks, sizes log-uniform)
  n, p, eps (0: opening angle alone), theta, n_leaf, soft, guard, precision,
  sphere (expansion centres of the bounding sphere instead of the centre of
  mass).
"""
import math

import numpy as np
import torch

import fmms_amd as fa

DEV = "cuda"
F8 = torch.float64


def _case(entry, model, n, p, n_leaf, eps=0.0, theta=1.0, soft=0.0, guard=0.0, precision="fp64",
          sphere=False, steps=0, refresh=1, graph=False, dt=0.0, systems=0, targets=0, chunk=32,
          name=None):
    c = dict(entry=entry, model=model, n=int(n), p=p, n_leaf=n_leaf, eps=eps, theta=theta,
             soft=soft, guard=guard, precision=precision, sphere=sphere, steps=steps,
             refresh=refresh, graph=graph, dt=dt, systems=systems, targets=targets, chunk=chunk)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small system through the reference's own interface (host arrays,
        # its default p, eps and leaf capacity): all latency
        _case("accel_host", "plummer", 1021, 8, 16, eps=1e-5, name="host_1k"),
        # a few steps of a small interactive simulation, tree rebuilt on each
        # (the integrator's own test parameters)
        _case("leapfrog", "plummer", 16381, 4, 16, eps=1e-3, steps=4, dt=1e-3,
              name="steps_16k"),
        # 100k softened bodies at the opening-angle MAC
        _case("accel", "plummer", 100000, 8, 32, theta=0.5, soft=1e-3, name="plummer_100k"),
        # a high-accuracy check run: order 24, rotation M2L
        _case("accel", "plummer", 30011, 24, 64, theta=0.5, name="order24_30k"),
        # a galaxy re-evaluated on its tree, bounding-sphere centres
        _case("evaluate", "hernquist", 250007, 6, 24, eps=1e-4, sphere=True,
              name="sphere_250k"),
        # the reference's published configuration: 1M bodies, p = 8, eps = 1e-5,
        # leaf capacity 16, error-controlled MAC
        _case("accel", "plummer", 1000000, 8, 16, eps=1e-5, name="reference_1m"),
        # the same size in the mixed form at the opening-angle MAC
        _case("accel", "plummer", 1048576, 8, 64, theta=0.5, soft=1e-3, precision="fp32bulk",
              name="mixed_1m"),
        # the force check: 4096 sampled targets against every body
        _case("direct", "plummer", 1048576, 0, 0, soft=1e-3, targets=4096, name="direct_1m"),
        # a batch of independent systems, evaluated together
        _case("accel", "ensemble", 1500000, 8, 96, theta=0.45, soft=1e-3, guard=1e-4,
              precision="fp32bulk", systems=48, name="ensemble_48"),
        # halos in a unit cube, frozen steps replayed from a graph
        _case("leapfrog", "halos", 2097152, 8, 128, theta=0.5, soft=1e-4, guard=1e-4,
              precision="fp32bulk", steps=5, refresh=5, graph=True, dt=1e-4, name="halos_2m"),
        # the plain FP64 form on a large system
        _case("accel", "plummer", 8388608, 7, 96, theta=0.5, soft=1e-3, name="fp64_8m"),
        # the headline: 16M bodies, mixed form
        _case("accel", "plummer", 16777216, 7, 112, theta=0.5, soft=1e-3, precision="fp32bulk",
              chunk=64, name="mixed_16m"),
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) | 1


def draw(rng):
    kind = rng.choice(["reference", "reference", "host", "angle", "angle", "mixed", "mixed",
                       "steps", "halos", "ensemble", "evaluate", "order", "direct"])
    model = rng.choice(["plummer", "hernquist", "disk"])
    if kind == "host":
        return _case("accel_host", model, _log_int(rng, 500, 200000), rng.randint(4, 9),
                     rng.choice([16, 24, 32]), eps=10.0 ** rng.uniform(-5, -3))
    if kind == "reference":
        return _case("accel", model, _log_int(rng, 2000, 600000), rng.randint(4, 10),
                     rng.choice([8, 16, 24, 32]), eps=10.0 ** rng.uniform(-5, -3),
                     sphere=rng.random() < 0.25)
    if kind == "angle":
        return _case("accel", model, _log_int(rng, 2000, 4000000), rng.randint(4, 10),
                     rng.choice([32, 48, 64, 96, 128]), theta=rng.uniform(0.4, 0.6),
                     soft=rng.choice([0.0, 1e-3]), chunk=rng.choice([16, 32, 64]))
    if kind == "mixed":
        return _case("accel", model, _log_int(rng, 2000, 8000000), rng.randint(6, 10),
                     rng.choice([32, 64, 96, 112, 128]), theta=rng.uniform(0.4, 0.6),
                     soft=rng.choice([0.0, 1e-3]), precision="fp32bulk",
                     chunk=rng.choice([16, 32, 64]))
    if kind == "steps":
        return _case("leapfrog", rng.choice(["plummer", "hernquist"]), _log_int(rng, 2000, 200000),
                     rng.choice([4, 6, 8]), rng.choice([16, 32]), eps=10.0 ** rng.uniform(-4, -3),
                     steps=rng.randint(2, 6), refresh=rng.choice([1, 2, 4]), dt=1e-3,
                     graph=rng.random() < 0.5)
    if kind == "halos":
        return _case("leapfrog", "halos", _log_int(rng, 100000, 2000000), 8,
                     rng.choice([64, 96, 128]), theta=0.5, soft=1e-4, guard=1e-4,
                     precision=rng.choice(["fp64", "fp32bulk"]), steps=rng.randint(2, 6),
                     refresh=rng.choice([4, 10]), graph=True, dt=1e-4)
    if kind == "ensemble":
        return _case("accel", "ensemble", _log_int(rng, 50000, 1500000), 8,
                     rng.choice([32, 64, 96]), theta=rng.choice([0.4, 0.45, 0.5]), soft=1e-3,
                     guard=1e-4, precision=rng.choice(["fp64", "fp32bulk"]),
                     systems=rng.randint(3, 64))
    if kind == "evaluate":
        return _case("evaluate", model, _log_int(rng, 5000, 300000), rng.randint(4, 9),
                     rng.choice([16, 24, 32]), eps=10.0 ** rng.uniform(-5, -3),
                     sphere=rng.random() < 0.5)
    if kind == "order":
        return _case("accel", "plummer", _log_int(rng, 3000, 30000), rng.choice([12, 16, 20, 24]),
                     rng.choice([32, 64]), theta=0.5)
    return _case("direct", model, _log_int(rng, 20000, 1000000), 0, 0,
                 soft=rng.choice([0.0, 1e-3]), targets=_log_int(rng, 64, 4096))


# ------------------------------------------------------------------- bodies
def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=F8)


def _directions(g, n):
    z = 2.0 * _rand(g, n) - 1.0
    a = 2.0 * math.pi * _rand(g, n)
    s = torch.sqrt(1.0 - z * z)
    return torch.stack([s * torch.cos(a), s * torch.sin(a), z], 1)


def _tangent(g, u):
    """Unit vectors at random angles across the unit vectors u."""
    w = torch.linalg.cross(u, _directions(g, u.shape[0]))
    return w / torch.linalg.vector_norm(w, dim=1, keepdim=True).clamp(min=1e-12)


def _sphere(g, model, n):
    """(position, velocity) of n bodies of total mass 1 on circular orbits."""
    if model == "plummer":  # scale 1, radii up to 20
        m = _rand(g, n) * (20.0 ** 3 / (1.0 + 20.0 ** 2) ** 1.5)
        m = m.clamp(min=1e-12)
        r = 1.0 / torch.sqrt(m ** (-2.0 / 3.0) - 1.0)
    else:  # Hernquist, scale 1, radii up to 100
        m = _rand(g, n) * (100.0 / 101.0) ** 2
        s = torch.sqrt(m.clamp(min=1e-12))
        r = s / (1.0 - s)
    u = _directions(g, n)
    return r[:, None] * u, torch.sqrt(m / r)[:, None] * _tangent(g, u)


def _disk(g, n):
    """Exponential disk, scale length 1, height 0.05, radii up to 10."""
    k = n + n // 50 + 64
    r = -torch.log(_rand(g, k).clamp(min=1e-12) * _rand(g, k).clamp(min=1e-12))
    r = r[r <= 10.0][:n]
    a = 2.0 * math.pi * _rand(g, n)
    z = 0.05 * torch.atanh((2.0 * _rand(g, n) - 1.0) * (1.0 - 1e-9))
    return torch.stack([r * torch.cos(a), r * torch.sin(a), z], 1)


def _halos(g, n):
    """64 Hernquist halos with 90 % of the bodies in a uniform unit cube."""
    w = 10.0 ** (2.0 * _rand(g, 64))
    w = w / w.sum()
    scale = 0.01 * 10.0 ** _rand(g, 64)
    cen = _rand(g, 64, 3)
    nh = int(0.9 * n + 0.5)
    edge = torch.round(torch.cumsum(w, 0) * nh)
    h = torch.searchsorted(edge, torch.arange(nh, device=DEV, dtype=F8), right=True).clamp(max=63)
    s = torch.sqrt((_rand(g, nh) * (20.0 / 21.0) ** 2).clamp(min=1e-12))
    r = scale[h] * s / (1.0 - s)
    u = _directions(g, nh)
    pos = torch.cat([cen[h] + r[:, None] * u, _rand(g, n - nh, 3)])
    v = torch.sqrt(0.9 * w[h] * s * s / r)
    vel = torch.cat([v[:, None] * _tangent(g, u), torch.zeros(n - nh, 3, device=DEV, dtype=F8)])
    return pos, vel


def _sizes(case):
    """Body counts of an ensemble's systems: log-uniform over a factor of 256."""
    k = case["systems"]
    w = 256.0 ** ((np.arange(k) * 0.6180339887498949) % 1.0)
    s = np.maximum(8, (w / w.sum() * case["n"]).astype(np.int64))
    s[-1] += case["n"] - s.sum()
    return s


def _bodies(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    n, model = case["n"], case["model"]
    if model == "ensemble":
        sizes = _sizes(case)
        pos = torch.cat([_disk(g, int(k)) if i % 2 else _sphere(g, "plummer", int(k))[0]
                         for i, k in enumerate(sizes)])
        mass = torch.cat([torch.full((int(k),), 1.0 / k, device=DEV, dtype=F8) for k in sizes])
        return pos, torch.zeros_like(pos), mass
    if model == "halos":
        pos, vel = _halos(g, n)
    elif model == "disk":
        pos = _disk(g, n)
        vel = torch.zeros_like(pos)
    else:
        pos, vel = _sphere(g, model, n)
    return pos, vel, torch.full((n,), 1.0 / n, device=DEV, dtype=F8)


# ---------------------------------------------------------------- the passes
def _context(case):
    return fa.Fmm(None, None, p=case["p"], eps=case["eps"] or math.inf, n_leaf=case["n_leaf"],
                  center_mode=fa.CenterMode.Sphere if case["sphere"] else fa.CenterMode.Com,
                  theta_max=case["theta"], softening=case["soft"], soft_mac=case["guard"],
                  precision=case["precision"], m2l_chunk=case["chunk"])


def _targets(case, seed):
    return fa.sample_ids(case["n"], case["targets"], seed + 1)


def prepare(case, seed):
    pos, vel, mass = _bodies(case, seed)
    n = case["n"]
    st = {"case": case, "n": n}
    if case["entry"] in ("accel_host", "direct"):
        st["pos"], st["mass"] = pos.cpu().numpy(), mass.cpu().numpy()
        if case["entry"] == "direct":
            st["ids"] = _targets(case, seed)
            return st
    else:
        st["pos"], st["mass"] = pos.contiguous(), mass
        st["acc"], st["pot"] = torch.empty_like(st["pos"]), torch.empty_like(mass)
    st["fmm"] = _context(case)
    if case["model"] == "ensemble":
        st["fmm"].set_systems(_sizes(case))
    torch.cuda.synchronize()
    if case["entry"] == "evaluate":
        st["fmm"].build_device(n, st["pos"].data_ptr(), mass.data_ptr())
    if case["entry"] == "leapfrog":
        st["vel"], st["started"] = vel.contiguous(), False
    return st


def run(st):
    c, n = st["case"], st["n"]
    if c["entry"] == "direct":
        acc, pot, f = fa.direct_sampled(st["pos"], st["mass"], st["ids"], softening=c["soft"])
        return {"accel": acc, "pot": pot, "f": f}
    if c["entry"] == "accel_host":
        r = st["fmm"].accel(st["pos"], st["mass"])
        return {"accel": r.accel, "pot": r.pot, "cells": r.n_cells}
    ptr = [st[k].data_ptr() for k in ("pos", "mass", "acc", "pot")]
    if c["entry"] == "leapfrog":  # each pass goes on from where the last one ended
        t = st["fmm"].leapfrog_device(n, ptr[0], st["vel"].data_ptr(), ptr[1], ptr[2], ptr[3],
                                      c["dt"], c["steps"], refresh_every=c["refresh"],
                                      acc_valid=st["started"], graph=c["graph"])
        st["started"] = True
        return {"pos": st["pos"], "vel": st["vel"], "accel": st["acc"], "pot": st["pot"], "t": t}
    if c["entry"] == "evaluate":
        st["fmm"].evaluate_device(n, *ptr)
    else:
        st["fmm"].accel_device(n, *ptr)
    return {"accel": st["acc"], "pot": st["pot"], "cells": st["fmm"].n_cells}


def work(case):
    """Bodies in and forces out; 22 operations per near pair and 8 T(p) per
    directed M2L pair. The pair counts are those of a Plummer sphere at
    theta = 0.5 (about 47 n_leaf near pairs and 1850 / n_leaf M2L pairs per
    body), scaled with the opening angle's volume; the error-controlled MAC
    counts as 0.6."""
    n = case["n"]
    if case["entry"] == "direct":
        return {"bytes": 32 * n + 44 * case["targets"], "flops": 22 * n * case["targets"]}
    p, leaf = case["p"], case["n_leaf"]
    v = (0.5 / (0.6 if case["eps"] else case["theta"])) ** 3
    t = sum((2 * k + 1) * (p - k + 1) ** 2 for k in range(p + 1))
    near = min(47.0 * leaf * v, float(n))
    flops = n * (22.0 * near + 8.0 * t * min(1850.0 / leaf * v, n / leaf))
    passes = max(1, case["steps"])
    io = 112 if case["entry"] == "leapfrog" else 64
    return {"bytes": io * n * passes, "flops": flops * passes}


# ------------------------------------------------------------- the direct sum
def _direct(pos, mass, soft, targets=None, block=1 << 24):
    """(accel, pot, sum m / r^2) at the target bodies (all: None), FP64."""
    n = pos.shape[0]
    tg = torch.arange(n, device=DEV) if targets is None else targets
    acc, pot, f = torch.empty(len(tg), 3, device=DEV, dtype=F8), [], []
    step = max(1, block // n)
    x, y, z = (pos[:, k].contiguous() for k in range(3))
    for a in range(0, len(tg), step):
        t = tg[a:a + step]
        dx, dy, dz = x[None] - x[t][:, None], y[None] - y[t][:, None], z[None] - z[t][:, None]
        r2 = dx * dx + dy * dy + dz * dz + soft * soft
        r2[torch.arange(len(t), device=DEV), t] = 1.0
        m = mass[None].expand(len(t), n).clone()
        m[torch.arange(len(t), device=DEV), t] = 0.0
        inv = r2.rsqrt()
        pm = m * inv
        pot.append(pm.sum(1))
        fm = pm * inv
        f.append(fm.sum(1))
        s = fm * inv
        acc[a:a + len(t), 0] = (s * dx).sum(1)
        acc[a:a + len(t), 1] = (s * dy).sum(1)
        acc[a:a + len(t), 2] = (s * dz).sum(1)
    return acc, torch.cat(pot), torch.cat(f)


def exact(case, seed):
    n = case["n"]
    if case["entry"] == "direct":
        pos, _, mass = _bodies(case, seed)
        ids = torch.from_numpy(_targets(case, seed).astype(np.int64)).to(DEV)
        acc, pot, f = _direct(pos, mass, case["soft"], ids)
        return {"accel": acc, "pot": pot, "f": f}
    evals = case["steps"] + 1 if case["entry"] == "leapfrog" else 1
    if case["model"] == "ensemble":
        sizes = _sizes(case)
        if float((sizes.astype(float) ** 2).sum()) > 7e10:
            return None
        pos, _, mass = _bodies(case, seed)
        got, a = [], 0
        for k in sizes:
            got.append(_direct(pos[a:a + k], mass[a:a + k], case["soft"])[:2])
            a += k
        return {"accel": torch.cat([g[0] for g in got]), "pot": torch.cat([g[1] for g in got]),
                "cells": None}
    if float(n) * n * evals > 7e10:
        return None
    pos, vel, mass = _bodies(case, seed)
    acc, pot, _ = _direct(pos, mass, case["soft"])
    if case["entry"] != "leapfrog":
        return {"accel": acc, "pot": pot, "cells": None}
    dt = case["dt"]
    for _ in range(case["steps"]):
        vel = vel + acc * (0.5 * dt)
        pos = pos + vel * dt
        acc, pot, _ = _direct(pos, mass, case["soft"])
        vel = vel + acc * (0.5 * dt)
    return {"pos": pos, "vel": vel, "accel": acc, "pot": pot, "t": dt * case["steps"]}

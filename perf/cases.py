"""Measured workloads of the diffusion-decay library, one pass per case.

A case is a stretch of a simulation as a program of this library runs it:
diffusion-decay steps at dt = 0.01 min with the agents' secretion and uptake,
and the field read back at the end of the stretch (a save).  Four kinds:

* "steps":   ``step(dt, n)`` on one resident microenvironment, then a save;
* "loop":    the main loop's own pair per step (``simulate_diffusion_decay``,
             ``simulate_cell_sources_and_sinks``, with ``bulk`` also
             ``simulate_bulk_sources_and_sinks``), then a save;
* "cells":   intervals of 10 steps between which the cells move: agent state
             up, steps, gradients at the cells back (chemotaxis), then a save;
* "batch":   many small microenvironments of different shapes advanced
             together, then every member saved.

Fields are FP64 or FP32 on the device; a save of an FP32 run is written in
single precision.  Kernel shapes are the library's own defaults.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DT, DX = 0.01, 20.0
W = DX ** 3


def _pkg():
    name = "physicellx_amd"
    if name not in sys.modules:
        here = os.path.join(ROOT, "physicell-x_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(here, "__init__.py"),
                                                      submodule_search_locations=[here])
        sys.modules[name] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _case(name, kind, nx, ny, nz, ns, precision, steps, agents, start="noise", faces="all",
          solver="blocking", planes=False, track=False, bulk=False, members=0):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, ns=ns, precision=precision, steps=steps,
                agents=agents, start=start, faces=faces, solver=solver, planes=planes, track=track,
                bulk=bulk, members=members)


def listed():
    return [
        # a unit-test-sized domain, one mechanics interval: all latency
        _case("tiny-fp64", "steps", 24, 20, 28, 2, "fp64", 10, 64),
        # a 1 mm domain of 20 um voxels, the usual size of a single-machine model
        _case("domain-50-fp64", "steps", 50, 50, 50, 1, "fp64", 60, 1000, start="fill"),
        # the same pair of calls per step as the reference's main loop makes,
        # totals of internalised substrate kept per cell
        _case("loop-64-fp64", "loop", 64, 64, 64, 2, "fp64", 30, 2000, track=True),
        # moving, chemotactic cells in a 1.5 mm domain
        _case("cells-75-fp32", "cells", 75, 75, 75, 2, "fp32", 60, 5000, start="fill"),
        # an ordinary larger run, one simulated minute
        _case("domain-100-fp64", "steps", 100, 100, 100, 2, "fp64", 100, 10000),
        # face values that differ from voxel to voxel, bulk supply and uptake
        _case("planes-bulk-fp64", "loop", 128, 96, 112, 1, "fp64", 30, 3000, planes=True, bulk=True),
        # ragged domains, some faces held and some substrates free, both solvers
        _case("ragged-fp32", "steps", 203, 157, 121, 3, "fp32", 100, 8000, faces="mixed", solver="avx256d"),
        _case("ragged-fp64", "steps", 131, 257, 67, 2, "fp64", 100, 5000, faces="mixed"),
        # an ensemble: edges 32 to 160, one to four substrates, three minutes
        _case("batch-24-fp32", "batch", 32, 32, 160, 4, "fp32", 300, 1000, start="fill", members=24),
        # the headline workload, a phenotype interval in single precision ...
        _case("cube-400-fp32", "steps", 400, 400, 400, 4, "fp32", 600, 100000),
        # ... and two simulated minutes in double
        _case("cube-400-fp64", "steps", 400, 400, 400, 4, "fp64", 200, 100000),
        # the largest domain: a million cells in a spheroid, half a minute
        _case("spheroid-800-fp64", "steps", 800, 800, 800, 2, "fp64", 50, 1000000, start="fill"),
    ]


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "loop", "cells", "batch"])
    prec = rng.choice(["fp64", "fp32"])
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    if kind == "batch":
        lo = log(16, 64)
        return {k: v for k, v in _case("", kind, lo, lo, log(64, 180), rng.randint(1, 4), prec, rng.randint(50, 300),
                                       1000, start="fill", members=rng.randint(4, 24)).items() if k != "name"}
    ns = rng.choice([1, 1, 2, 2, 3, 4, 6, 8])
    while True:
        edges = [log(12, 640) for _ in range(3)]
        n = edges[0] * edges[1] * edges[2]
        if n * ns <= 1.6e8 and (kind == "steps" or n * ns <= 2e7):
            break
    steps = rng.choice([10, 30, 60, 100])
    return {k: v for k, v in _case(
        "", kind, *edges, ns, prec, steps, max(1, min(200000, int(n * 10 ** rng.uniform(-4, -2)))),
        start="noise" if n * ns < 4e7 else "fill", faces=rng.choice(["all", "all", "mixed", "none"]),
        solver=rng.choice(["blocking", "blocking", "avx256d"]),
        planes=kind == "loop" and rng.random() < 0.3, track=kind != "cells" and rng.random() < 0.2,
        bulk=kind == "loop" and rng.random() < 0.3).items() if k != "name"}


# ---- inputs, from the seed alone -------------------------------------------------

def _agents(rng, c, n):
    """Cells of 2494 um^3 with secretion and uptake rates up to 10 /min
    towards a saturation density of 40; a few share a voxel."""
    na, ns = c["agents"], c["ns"]
    nx, ny, nz = n
    if na >= 500000:  # a rim-weighted spheroid filling three quarters of the domain
        r = np.clip(1 - np.abs(rng.normal(0, 0.15, na)), 0, 1) * 0.375 * min(n)
        v = rng.normal(size=(na, 3))
        v *= (r / np.linalg.norm(v, axis=1))[:, None]
        ijk = np.clip((v + np.array(n) / 2).astype(np.int64), 0, np.array(n) - 1)
    else:
        ijk = np.stack([rng.integers(0, m, na) for m in n], 1)
    voxel = ((ijk[:, 0] * ny + ijk[:, 1]) * nz + ijk[:, 2]).astype(np.int32)
    S, U = rng.uniform(0, 10, (na, ns)), rng.uniform(0, 10, (na, ns))
    E = rng.uniform(0, 5, (na, ns))
    return voxel, ijk, S, U, E


def _constants(S, U, E):
    f = DT * 2494.0 / W
    return S * 40.0 * f, 1.0 + f * S + f * U, E * DT / W, E * DT


def _one(rng, c, n, ns):
    """Everything of one microenvironment but its field."""
    p = dict(n=n, ns=ns, D=10 ** rng.uniform(3, 5, ns), decay=rng.uniform(0.01, 1.0, ns))
    base = rng.uniform(0, 40, ns)
    p["base"] = base
    p["act"], p["reg"] = np.ones(ns, np.uint8), np.ones(6, np.uint8)
    p["fv"] = np.tile(base, (6, 1))
    if c["faces"] == "mixed":
        p["act"] = (np.arange(ns) % 2 == 0).astype(np.uint8)
        p["reg"] = np.array([1, 0, 1, 1, 0, 1], np.uint8)
        p["fv"] = rng.uniform(0, 40, (6, ns))
    elif c["faces"] == "none":
        p["act"], p["reg"] = np.zeros(ns, np.uint8), np.zeros(6, np.uint8)
    return p


def _shapes(c):
    """The members' edges (nx..nz of the case) and substrate counts: part of
    the case, not of its inputs."""
    rng = np.random.default_rng(c["members"])
    return [(tuple(int(v) for v in rng.integers(c["nx"], c["nz"] + 1, 3)), int(rng.integers(1, c["ns"] + 1)))
            for _ in range(c["members"])]


def _inputs(c, seed):
    rng = np.random.default_rng(seed)
    if c["kind"] == "batch":
        got = []
        for n, ns in _shapes(c):
            p = _one(rng, c, n, ns)
            p["voxel"], _, S, U, E = _agents(rng, dict(c, ns=ns, agents=max(1, n[0] * n[1] * n[2] // c["agents"])), n)
            p["c1"], p["c2"], p["e2"], p["e1"] = _constants(S, U, E)
            got.append(p)
        return got
    n = (c["nx"], c["ny"], c["nz"])
    p = _one(rng, c, n, c["ns"])
    p["voxel"], ijk, p["S"], p["U"], p["E"] = _agents(rng, c, n)
    p["c1"], p["c2"], p["e2"], p["e1"] = _constants(p["S"], p["U"], p["E"])
    if c["kind"] == "cells":  # a random walk of about a third of a voxel per interval
        pos = (ijk + rng.uniform(0, 1, ijk.shape)) * DX
        top = np.array(n) * DX * (1 - 1e-12)
        p["pos"] = []
        for _ in range(c["steps"] // 10):
            p["pos"].append(pos.copy())
            pos = np.clip(pos + rng.normal(0, 7.0, pos.shape), 0, top)
        ijks = [np.minimum((q / DX).astype(np.int64), np.array(n) - 1) for q in p["pos"]]
        p["vox"] = [((q[:, 0] * n[1] + q[:, 1]) * n[2] + q[:, 2]).astype(np.int32) for q in ijks]
    if c["planes"]:  # the boundary values vary along the faces: one value per voxel
        i, j, k = (np.arange(m)[:, None] for m in n)
        a, b, g = (rng.uniform(0.1, 0.4, c["ns"])[None, :] for _ in range(3))
        fx, fy, fz = (p["base"] + 0.5) * np.cos(a * i / n[0] * 8), np.sin(b * j / n[1] * 8), np.cos(g * k / n[2] * 8)
        yz = lambda x: (x + fy[:, None, :] + fz[None, :, :])  # noqa: E731
        xz = lambda y: (fx[:, None, :] + y + fz[None, :, :])  # noqa: E731
        xy = lambda z: (fx[:, None, :] + fy[None, :, :] + z)  # noqa: E731
        p["planes"] = [yz(fx[0]), yz(fx[-1]), xz(fy[0]), xz(fy[-1]), xy(fz[0]), xy(fz[-1])]
    if c["bulk"]:
        N = n[0] * n[1] * n[2] * c["ns"]
        p["bS"], p["bT"], p["bU"] = rng.uniform(0, 0.2, N), rng.uniform(20, 40, N), rng.uniform(0, 0.1, N)
    return p


def _field(c, seed, p):
    """The initial field [ns][nz][ny][nx] (device order): the boundary value
    of each substrate plus noise; None where it starts uniform."""
    if c["start"] == "fill":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) + 1)
    nx, ny, nz = p["n"]
    u = torch.empty((p["ns"], nz, ny, nx), dtype=torch.float64, device=dev)
    u.normal_(generator=g)
    return u.add_(torch.from_numpy(p["base"]).to(dev)[:, None, None, None])


def prepare(case, seed):
    c, pk = case, _pkg()
    p = _inputs(c, seed)
    if c["kind"] == "batch":
        b = pk.Batch(c["precision"])
        ids = []
        for m in p:
            i = b.add(*m["n"], m["ns"], DX, m["D"], m["decay"], m["act"], m["reg"], m["fv"])
            b.fill(i, m["base"])
            b.set_agents(i, m["voxel"], m["c1"], m["c2"], m["e2"])
            ids.append(i)
        return dict(c=c, batch=b, ids=ids)
    e = pk.Microenvironment(*p["n"], p["ns"], DX, c["precision"])
    e.set_coefficients(p["D"], p["decay"])
    e.set_dirichlet(p["act"], p["reg"], p["fv"])
    if c["planes"]:
        e.set_dirichlet_planes(p["planes"])
    e.set_solver(c["solver"])
    u = _field(c, seed, p)
    if u is None:
        e.fill(p["base"])
    else:
        e.upload(u.cpu().numpy().reshape(-1), "soa")
        del u
        torch.cuda.empty_cache()
    if c["kind"] != "cells":
        e.set_agents(p["voxel"], p["c1"], p["c2"], p["e2"])
        if c["track"]:
            e.track_internalized(None, p["e1"])
    if c["bulk"]:
        e.set_bulk_rates(p["bS"], p["bT"], p["bU"])
    s = dict(c=c, env=e, box=np.array([0.0, 0.0, 0.0, *(m * DX for m in p["n"])]))
    # the program's save buffers
    count = p["n"][0] * p["n"][1] * p["n"][2] * p["ns"]
    s["field"] = torch.zeros(count, dtype=torch.float64)
    s["single"] = torch.zeros(count, dtype=torch.float32) if c["precision"] == "fp32" else None
    if c["kind"] == "cells":
        s["V"], s["sat"] = np.full(c["agents"], 2494.0), np.full((c["agents"], p["ns"]), 40.0)
        for k in ("S", "U", "E", "pos", "vox"):
            s[k] = p[k]
    return s


def run(state):
    s, c = state, state["c"]
    if c["kind"] == "batch":
        b = s["batch"]
        b.step(DT, c["steps"])
        out = [b.download(i, "soa") for i in s["ids"]]
        return [f.astype(np.float32) for f in out] if c["precision"] == "fp32" else out
    e, out = s["env"], {}
    if c["kind"] == "steps":
        e.step(DT, c["steps"])
    elif c["kind"] == "loop":
        for _ in range(c["steps"]):
            if c["bulk"]:
                e.simulate_bulk_sources_and_sinks(DT)
            e.simulate_diffusion_decay(DT)
            e.simulate_cell_sources_and_sinks()
    else:
        grads = []
        for pos, vox in zip(s["pos"], s["vox"]):
            e.set_agents_state(pos, s["box"], s["V"], s["S"], s["U"], s["E"], s["sat"], DT)
            e.step(DT, 10)
            grads.append(e.gradients_at(vox))
        out["gradients"] = np.stack(grads).astype(np.float32 if c["precision"] == "fp32" else np.float64)
    e.download("soa", out=s["field"].numpy())
    if c["precision"] == "fp32":
        s["single"].copy_(s["field"])
    out["field"] = s["single"] if c["precision"] == "fp32" else s["field"]
    if c["track"]:
        out["internalized"] = e.internalized().astype(np.float32 if c["precision"] == "fp32" else np.float64)
    return out


def work(case):
    """Per step the field is read and written once (the steps follow one
    another), the agents' constants are read once; the save reads the field
    once and writes it to the host.  Per value and axis the line solve takes
    about five operations."""
    c = case
    b = 8 if c["precision"] == "fp64" else 4
    if c["kind"] == "batch":
        vals = sum(n[0] * n[1] * n[2] * ns for n, ns in _shapes(c))
        agents = vals / c["agents"]
    else:
        vals = c["nx"] * c["ny"] * c["nz"] * c["ns"]
        agents = c["agents"] * c["ns"]
    per = 2 * vals * b + agents * (24 + 2 * b)
    if c["bulk"]:
        per += vals * 16
    if c["track"]:
        per += agents * 24
    return {"bytes": c["steps"] * per + vals * 2 * b, "flops": c["steps"] * (15 * vals + 3 * agents)}


# ---- the same in 64 bits, dense operators on whole axes ---------------------------

def _inverse(n, D, decay, dev):
    """The inverse of one axis matrix: diagonal 1 + 2 c1 + c2 (one c1 less at
    each end), off-diagonals -c1."""
    c1, c2 = D * DT / DX / DX, decay * DT / 3.0
    m = torch.zeros((n, n), dtype=torch.float64, device=dev)
    i = torch.arange(n, device=dev)
    m[i, i] = 1 + 2 * c1 + c2
    m[0, 0] -= c1
    m[n - 1, n - 1] -= c1
    m[i[1:], i[:-1]] = m[i[:-1], i[1:]] = -c1
    return torch.linalg.inv(m)


def _apply_faces(u, p, d):
    """u [nz][ny][nx] of substrate d: every boundary voxel takes its value."""
    if not p["act"][d]:
        return
    if "planes" in p:
        t = [torch.as_tensor(np.ascontiguousarray(q[..., d]), device=u.device) for q in p["planes"]]
        u[:, :, 0], u[:, :, -1] = t[0].T, t[1].T
        u[:, 0, :], u[:, -1, :] = t[2].T, t[3].T
        u[0], u[-1] = t[4].T, t[5].T
        return
    side = [u[:, :, 0], u[:, :, -1], u[:, 0, :], u[:, -1, :], u[0], u[-1]]
    for f in range(6):
        side[f].fill_(1.0)
    for f in range(6):  # the last registered face wins
        if p["reg"][f]:
            side[f].fill_(float(p["fv"][f, d]))


def _rounds(voxel, n, dev):
    """Agents in rounds of distinct voxels, in agent order within a voxel:
    (flat device-order positions, agent indices) per round."""
    nx, ny, nz = n
    v = voxel.astype(np.int64)
    at = (v % nz * ny + v // nz % ny) * nx + v // (nz * ny)
    order = np.argsort(at, kind="stable")
    srt = at[order]
    first = np.r_[True, srt[1:] != srt[:-1]]
    rank = np.arange(len(srt)) - np.maximum.accumulate(np.where(first, np.arange(len(srt)), 0))
    return [(torch.from_numpy(srt[rank == r]).to(dev), torch.from_numpy(order[rank == r]).to(dev))
            for r in range(int(rank.max()) + 1)]


def _diffuse(u, inv, p, d, solver):
    nz, ny, nx = u.shape
    _apply_faces(u, p, d)
    u = torch.matmul(u.reshape(-1, nx), inv[0].T).reshape(nz, ny, nx)
    _apply_faces(u, p, d)
    u = torch.matmul(inv[1], u)
    _apply_faces(u, p, d)
    u = torch.matmul(inv[2], u.reshape(nz, -1)).reshape(nz, ny, nx)
    if solver == "blocking":
        _apply_faces(u, p, d)
    return u


def _gradient_at(u, vox, n):
    nx, ny, nz = n
    v = torch.from_numpy(vox.astype(np.int64)).to(u.device)
    k, j, i = v % nz, v // nz % ny, v // (nz * ny)
    out = []
    for axis, (pos, m) in enumerate(((i, nx), (j, ny), (k, nz))):
        if m == 1:
            out.append(torch.zeros(len(v), dtype=torch.float64, device=u.device))
            continue
        lo, hi = (pos - 1).clamp(min=0), (pos + 1).clamp(max=m - 1)
        at = lambda q: u[(k, j, q) if axis == 0 else (k, q, i) if axis == 1 else (q, j, i)]  # noqa: E731
        out.append((at(hi) - at(lo)) / ((hi - lo).double() * DX))
    return torch.stack(out, 1)


def _solve(c, p, field, dev):
    """Final fields [ns][nz][ny][nx], gradients per interval, internalised totals."""
    n, ns, na = p["n"], p["ns"], len(p["voxel"])
    nx, ny, nz = n
    fields, grads, inner = [], [], torch.zeros((na, ns), dtype=torch.float64, device=dev)
    fixed = _rounds(p["voxel"], n, dev) if c["kind"] != "cells" else None
    moving = [_rounds(v, n, dev) for v in p["vox"]] if c["kind"] == "cells" else None
    for d in range(ns):
        inv = [_inverse(m, p["D"][d], p["decay"][d], dev) for m in n]
        u = field[d].clone() if field is not None else torch.full((nz, ny, nx), float(p["base"][d]),
                                                                   dtype=torch.float64, device=dev)
        c1, c2, e2, e1 = (torch.from_numpy(np.ascontiguousarray(p[q][:, d])).to(dev) for q in ("c1", "c2", "e2", "e1"))
        if c["bulk"]:
            S, T, U = (torch.from_numpy(p[q]).to(dev).reshape(nx, ny, nz, ns)[..., d].permute(2, 1, 0).contiguous()
                       for q in ("bS", "bT", "bU"))
        mine = []
        for step in range(c["steps"]):
            if c["bulk"]:
                u = (u + DT * (T * S)) / (1 + DT * (U + S))
            u = _diffuse(u, inv, p, d, c["solver"])
            flat = u.reshape(-1)
            for at, a in (fixed if fixed is not None else moving[step // 10]):
                rho = flat[at]
                if c["track"]:
                    inner[a, d] -= W * ((1 - c2[a]) * rho + c1[a]) / c2[a]
                    inner[a, d] -= e1[a]
                flat[at] = (rho + c1[a]) / c2[a] + e2[a]
            if moving is not None and step % 10 == 9:
                mine.append(_gradient_at(u, p["vox"][step // 10], n))
        fields.append(u)
        grads.append(mine)
    g = torch.stack([torch.stack([grads[d][t] for d in range(ns)], 1) for t in range(len(grads[0]))]) if moving else None
    return fields, g, inner


def exact(case, seed):
    c = case
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = _inputs(c, seed)
    if c["kind"] == "batch":
        return [torch.cat([u.reshape(-1) for u in _solve(c, m, None, dev)[0]]).cpu() for m in p]
    fields, grads, inner = _solve(c, p, _field(c, seed, p), dev)
    got = {"field": torch.cat([u.reshape(-1).cpu() for u in fields])}
    if c["kind"] == "cells":
        got["gradients"] = grads.cpu()
    if c["track"]:
        got["internalized"] = inner.cpu()
    return got

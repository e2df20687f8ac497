"""Performance cases of the multigrid Euler library: the solves its users run,
through the public entry points of the ``mgcfd`` binding.

Four forms of use, as the README and the benchmark name them:

  solve   one mesh declared through the OP2 interface (``mgcfd.Solver``) and
          advanced device-resident (``mgcfd_mg_run``), then its flow state
          fetched: what a program does that links the library for one solve;
  loops   the same mesh driven loop by loop (``op_par_loop_*``), as the
          reference's own driver and the bundled ``euler3d`` run it;
  batch   several meshes of uneven size concatenated in one context
          (``mgcfd.Batch``), or one large mesh, with every state fetched;
  serve   requests submitted to ``mgcfd.Server`` and polled until done, with
          the planning of each request's mesh inside the call.

Sizes span the repository's own workloads: 10K nodes (the smallest served
request) over the 40^3 box, the 300K-node / 930K-edge mesh and the 20K-500K
batch to the 1M-node shard and a 2M-node box.  A mesh's topology comes from
its size; the seed gives its dual-face areas, freestream and initial flow.
"""
import functools
import math
import os
import sys
import time

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mg-cfd-app-op2_amd"))

import mgcfd  # noqa: E402

GAMMA = 1.4


def listed():
    return [
        # smallest requests: a cycle is a chain of short dependent launches
        dict(name="solve-10k-default", kind="solve", mesh="knn", nodes=10007, levels=4, variant="gather_exact",
             cycles=20),
        # the 40^3 box solve of the reference's -g 10 runs, default flux
        dict(name="solve-box40-default", kind="solve", mesh="box", nodes=40 ** 3, levels=4, variant="gather_exact",
             cycles=10),
        # the 300K-node solve as a program gets it that chooses nothing
        dict(name="solve-300k-default", kind="solve", mesh="knn", nodes=300000, levels=4, variant="gather_exact",
             cycles=25),
        # ... and with the fastest FP64 and the mixed-precision flux (-g 50)
        dict(name="solve-300k-fp64", kind="solve", mesh="knn", nodes=300000, levels=4, variant="part_atomic",
             cycles=50),
        dict(name="solve-300k-mixed", kind="solve", mesh="knn", nodes=300000, levels=4, variant="mixed_atomic",
             cycles=50),
        # a mid-sized solve that has to repeat bit for bit
        dict(name="solve-100k-coloured", kind="solve", mesh="knn", nodes=100003, levels=4, variant="part_coloured",
             cycles=50),
        # loop by loop with host reductions, as the reference's driver runs
        dict(name="loops-30k-default", kind="loops", mesh="knn", nodes=30011, levels=4, variant="gather_exact",
             cycles=10),
        dict(name="loops-300k-fp64", kind="loops", mesh="knn", nodes=300000, levels=4, variant="part_atomic",
             cycles=10),
        # parameter studies: uneven meshes advanced together
        dict(name="batch-12-fp64", kind="batch", mesh="knn", meshes=12, nodes=20011, nodes_max=200003, levels=4,
             variant="part_atomic", cycles=30),
        dict(name="batch-24-mixed", kind="batch", mesh="knn", meshes=24, nodes=10007, nodes_max=50021, levels=4,
             variant="mixed_atomic", cycles=30),
        # one large solve: the working set exceeds every cache
        dict(name="large-1m-fp64", kind="batch", mesh="knn", meshes=1, nodes=1000000, nodes_max=1000000, levels=4,
             variant="part_atomic", cycles=40),
        # served requests, FP64 and mixed precision by turns, planning included
        dict(name="serve-8", kind="serve", mesh="knn", meshes=8, nodes=10007, nodes_max=60013, levels=4,
             variant="part_coloured", cycles=100),
    ]


def draw(rng):
    """A case of the same ranges; costs at most what the largest listed one does."""
    def log_int(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    kind = rng.choice(["solve", "solve", "solve", "loops", "batch", "batch", "serve"])
    fp64 = ["gather_exact", "gather_fast", "part_coloured", "part_atomic"]
    case = dict(kind=kind, levels=rng.choice([2, 3, 4, 4, 4]))
    if kind in ("solve", "loops"):
        nodes = log_int(8_000, 400_000 if kind == "solve" else 200_000)
        if rng.random() < 0.25:
            case.update(mesh="box", nodes=max(20, round(nodes ** (1 / 3))) ** 3)
        else:
            case.update(mesh="knn", nodes=nodes)
        most = 15_000_000 // case["nodes"]
        case.update(variant=rng.choice(fp64 + ["mixed_coloured", "mixed_atomic"]),
                    cycles=max(5, min(most, rng.randint(5, 60 if kind == "solve" else 12))))
    elif kind == "batch":
        top = log_int(20_000, 300_000)
        n = rng.randint(1, max(1, min(16, 800_000 // top)))
        case.update(mesh="knn", meshes=n, nodes=min(top, log_int(8_000, top)) if n > 1 else top, nodes_max=top,
                    variant=rng.choice(fp64 + ["mixed_coloured", "mixed_atomic"]), cycles=rng.randint(10, 40))
    else:
        top = log_int(12_000, 100_000)
        case.update(mesh="knn", meshes=rng.randint(2, 8), nodes=min(top, log_int(8_000, top)), nodes_max=top,
                    variant=rng.choice(["part_coloured", "mixed_coloured", "gather_exact"]),
                    cycles=rng.randint(30, 120))
    return case


# ----------------------------------------------------------------- meshes --

@functools.lru_cache(maxsize=64)
def base_mesh(kind, nodes, levels):
    if kind == "box":
        return mgcfd.mesh_box(round(nodes ** (1 / 3)), levels, seed=3)
    return mgcfd.mesh_knn(nodes, int(round(3.1 * nodes)), levels, seed=5)


def sizes(case):
    """Level-0 node counts of the case's meshes, spread over their logarithm."""
    n = case.get("meshes", 1)
    lo, hi = case["nodes"], case.get("nodes_max", case["nodes"])
    return [round(lo * (hi / lo) ** (i / max(1, n - 1))) if n > 1 else hi for i in range(n)]


def inputs(case, seed):
    """Per mesh: levels with the seed's dual-face areas, Mach number, angle."""
    out = []
    for i, n in enumerate(sizes(case)):
        rng = np.random.default_rng([seed, i])
        mesh = []
        for lv in base_mesh(case["mesh"], n, case["levels"]):
            lv = dict(lv)
            lv["edge_weights"] = lv["edge_weights"] * rng.uniform(0.9, 1.1, (len(lv["edge_weights"]), 1))
            mesh.append(lv)
        out.append((mesh, rng.uniform(0.3, 0.8), rng.uniform(-2.0, 6.0)))
    return out


def initial_flow(n, ffv, seed):
    """A disturbed freestream, 1% in each variable."""
    rng = np.random.default_rng([seed, 99])
    v = np.asarray(ffv)[None, :] * (1.0 + 0.01 * rng.uniform(-1, 1, (n, 5)))
    v[:, 3] += 0.01 * rng.uniform(-1, 1, n)
    return v


@functools.lru_cache(maxsize=1)
def runtime():
    return mgcfd.Runtime()


class Handle:
    """What a program keeps between calls: a solver, batch or server with its
    inputs.  Batches and servers are released with the last reference; a
    declared mesh lives as long as the library instance."""

    def __init__(self, case, thing, data=None):
        self.case, self.thing, self.data = case, thing, data

    def __del__(self):
        if not isinstance(self.thing, mgcfd.Solver):
            self.thing.close()


def variant_of(case, i):
    """Served requests alternate between the FP64 variant and mixed precision."""
    return case["variant"] if case["kind"] != "serve" or i % 2 == 0 else "mixed_coloured"


def prepare(case, seed):
    rt = runtime()
    data = inputs(case, seed)
    if case["kind"] in ("solve", "loops"):
        mesh, mach, aoa = data[0]
        s = mgcfd.Solver(rt, mesh, mach, aoa)
        s.setup()
        rt.upload(s.lv[0].variables, initial_flow(len(mesh[0]["coords"]), s.fs["ff_variable"], seed))
        return Handle(case, s)
    if case["kind"] == "batch":
        b = mgcfd.Batch(rt, [m for m, _, _ in data], [x for _, x, _ in data], [x for _, _, x in data],
                        case["variant"])
        return Handle(case, b)
    return Handle(case, mgcfd.Server(rt, max_active=8, chunk=case["cycles"]), data)


def run(state):
    case, x = state.case, state.thing
    if case["kind"] in ("solve", "loops"):
        # the flux variant and the freestream constants are the library
        # instance's: set to this solve's before it runs
        x.rt.set_flux_variant(mgcfd.FLUX_VARIANTS[case["variant"]])
        x.rt.decl_consts(x.fs)
        if case["kind"] == "solve":
            status, rms = x.run_device(case["cycles"])
        else:
            status, rms, _ = x.run_loops(case["cycles"])
        return dict(status=status, rms=np.asarray(rms), variables=x.state(0))
    if case["kind"] == "batch":
        status, rms = x.run(case["cycles"])
        return dict(status=status, rms=rms, variables=[x.fetch(i, 0) for i in range(x.n)])
    ids = [x.submit(m, mach, aoa, variant_of(case, i), max_cycles=case["cycles"])
           for i, (m, mach, aoa) in enumerate(state.data)]
    done = {}
    while len(done) < len(ids):
        x.progress()
        for i in ids:
            if i not in done:
                r = x.result(i)
                if r is not None:
                    done[i] = r
        time.sleep(0.0005)
    return dict(status=[done[i]["status"] for i in ids], rms=[done[i]["rms"] for i in ids],
                variables=[done[i]["variables"] for i in ids])


def work(case):
    """Per Runge-Kutta stage: the edges' weights and end points, the state
    read and written and the old state read; per smoothing step also the
    volumes, step factors and residuals; per transfer the fine and coarse
    states.  The flux of an edge is 201 operations as the reference writes
    it, a node's update about 30."""
    nbytes = flops = 0
    for n in sizes(case):
        mesh = base_mesh(case["mesh"], n, case["levels"])
        last = len(mesh) - 1
        for l, lv in enumerate(mesh):
            nodes, edges = len(lv["coords"]), len(lv["edge_to_node"])
            steps = 1 if l in (0, last) else 2
            nbytes += steps * (3 * (32 * edges + 120 * nodes) + 64 * nodes)
            flops += steps * 3 * (201 * edges + 30 * nodes)
            if l < last:        # restriction from, and prolongation to, this level
                coarse = len(mesh[l + 1]["coords"])
                nbytes += (44 * nodes + 40 * coarse) + (148 * nodes + 64 * coarse)
                flops += 5 * nodes + 25 * nodes
    return dict(bytes=nbytes * case["cycles"], flops=flops * case["cycles"])


# ------------------------------------------------------------- 64-bit truth --

class Level:
    """One level of the multigrid scheme in plain FP64 torch."""

    def __init__(self, lv, dev):
        t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)  # noqa: E731
        self.x = t(lv["coords"], torch.float64)
        e = t(lv["edge_to_node"], torch.int64)
        self.a, self.b = e[:, 0].contiguous(), e[:, 1].contiguous()
        w = t(lv["edge_weights"], torch.float64)
        d = self.x[self.b] - self.x[self.a]
        dist, area = d.square().sum(1).sqrt(), w.square().sum(1).sqrt()
        self.n = len(self.x)
        tet = dist * area / 6.0
        self.vol = torch.zeros(self.n, dtype=torch.float64, device=dev)
        self.vol.index_add_(0, self.a, tet).index_add_(0, self.b, tet)
        self.w = d / dist[:, None] * area[:, None] / dist[:, None] * 1e-7
        self.ewt = self.w.square().sum(1).sqrt()
        self.bn = t(lv["bnd_to_node"], torch.int64)
        group = t(lv["bnd_group"], torch.int64)
        bw = t(lv["bnd_weights"], torch.float64) * 1e-7
        self.wall = torch.where((group <= 2)[:, None], bw, torch.zeros_like(bw))
        self.far = torch.where(((group >= 3) & (group <= 7))[:, None], bw, torch.zeros_like(bw))
        self.up = None if lv.get("node_to_mg_node") is None else t(lv["node_to_mg_node"], torch.int64)
        self.flux = torch.zeros(self.n, 5, dtype=torch.float64, device=dev)


def thermo(u):
    vel = u[:, 1:4] / u[:, 0:1]
    ssq = vel.square().sum(1)
    p = (GAMMA - 1.0) * (u[:, 4] - 0.5 * u[:, 0] * ssq)
    return vel, ssq, p, (GAMMA * p / u[:, 0]).sqrt()


def tensors(u):
    """[n][5][3] convective fluxes and [n] wave speeds of a state."""
    vel, ssq, p, c = thermo(u)
    f = torch.empty(len(u), 5, 3, dtype=u.dtype, device=u.device)
    f[:, 0] = u[:, 1:4]
    f[:, 1:4] = u[:, 1:4, None] * vel[:, None, :]
    for k in range(3):
        f[:, 1 + k, k] += p
    f[:, 4] = vel * (u[:, 4] + p)[:, None]
    return f, ssq.sqrt() + c, p


def smooth(L, var, ff, sc):
    """One smoothing step: (new state, residual)."""
    old = var
    vel, ssq, p, c = thermo(var)
    dt = 0.5 * L.vol.pow(1.0 / 3.0) / (ssq.sqrt() + c)
    sf = dt.min() / L.vol
    for rk in range(3):
        f, s, p = tensors(var)
        diff = (-0.5 * sc) * (L.ewt * (s[L.a] + s[L.b]))[:, None] * (var[L.a] - var[L.b])
        inc = diff - 0.5 * ((f[L.a] + f[L.b]) * L.w[:, None, :]).sum(2)
        flux = L.flux if rk == 0 else torch.zeros_like(L.flux)
        flux = flux.index_add(0, L.a, inc).index_add_(0, L.b, -inc)
        bnd = 0.5 * ((ff[None] + f[L.bn]) * L.far[:, None, :]).sum(2)
        bnd[:, 1:4] += L.wall * p[L.bn][:, None]
        flux.index_add_(0, L.bn, bnd)
        var = old + (sf / (4 - rk))[:, None] * flux
    L.flux = torch.zeros_like(L.flux)
    return var, var - old


def solve64(mesh, mach, aoa, cycles, start, dev):
    """(RMS history, level-0 state) of the multigrid solve in FP64."""
    fs = mgcfd_free_state(mach, aoa)
    ffv = torch.tensor(fs, dtype=torch.float64, device=dev)[None]
    ff, _, _ = tensors(ffv)
    ff, sc = ff[0], float(np.float32(0.2))
    lv = [Level(m, dev) for m in mesh]
    var = [ffv.repeat(L.n, 1) for L in lv]
    if start is not None:
        var[0] = torch.as_tensor(start, device=dev)
    res, rms, last = [None] * len(lv), [], len(lv) - 1
    for _ in range(cycles):
        for l in range(len(lv)):
            if l:
                n = torch.zeros(lv[l].n, dtype=torch.float64, device=dev)
                n.index_add_(0, lv[l - 1].up, torch.ones(lv[l - 1].n, dtype=torch.float64, device=dev))
                total = torch.zeros_like(var[l]).index_add_(0, lv[l - 1].up, var[l - 1])
                var[l] = torch.where((n > 0)[:, None], total / n.clamp(min=1)[:, None], var[l])
            var[l], res[l] = smooth(lv[l], var[l], ff, sc)
            if l == 0:
                rms.append((res[0].square().sum() / lv[0].n).sqrt())
        for l in range(last - 1, -1, -1):
            up = lv[l].up
            d = (lv[l].x - lv[l + 1].x[up]).abs()
            dm = d.square().sum(1, keepdim=True).sqrt()
            var[l] = var[l] - torch.cat([dm, d, dm], 1) * (res[l + 1][up] - res[l])
            if l:
                var[l], res[l] = smooth(lv[l], var[l], ff, sc)
    return torch.stack(rms).cpu().numpy(), var[0].cpu().numpy()


def mgcfd_free_state(mach, aoa_deg):
    """Conserved variables of the freestream: density 1.4, pressure 1."""
    a = math.radians(aoa_deg)
    return [1.4, 1.4 * mach * math.cos(a), 1.4 * mach * math.sin(a), 0.0, 1.4 * 0.5 * mach * mach + 1.0 / (GAMMA - 1.0)]


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    got = []
    for mesh, mach, aoa in inputs(case, seed):
        start = None
        if case["kind"] in ("solve", "loops"):
            start = initial_flow(len(mesh[0]["coords"]), mgcfd_free_state(mach, aoa), seed)
        got.append(solve64(mesh, mach, aoa, case["cycles"], start, dev))
    if case["kind"] in ("solve", "loops"):
        return dict(status=None, rms=got[0][0], variables=got[0][1])
    rms = [r for r, _ in got]
    return dict(status=None, rms=np.stack(rms) if case["kind"] == "batch" else rms, variables=[v for _, v in got])

"""The framework's work as its users have it do: the cases that its speed is measured on.

Every pass goes through the public Python API (or, for the search on device points, the C entry point the
API's binding exposes).  Rollouts start from an uploaded state, step it, and hand back the whole state: read
back to the host where a program draws or logs small groups, left on the device (arrays in storage order, with
the agent index of each slot) where it is large.  So a pass always does the same work, however often it runs.

Results are the same sequence of correctly rounded operations whatever kernels compute them, so every case
states "exact".
"""
import ctypes
import dataclasses
import math

import numpy as np
import torch

import gpusteer_amd as gs
from gpusteer_amd import _capi as capi
from gpusteer_amd import api, formats, scenarios
from gpusteer_amd.ensemble import Calibration, Ensemble, step_choke
from gpusteer_amd.plugins import ChokePointNew, MultiGroup
from gpusteer_amd.scenarios import FlockTerm
from gpusteer_amd.state import AGENT_FIELDS

# The flocking terms of the group plugin with explicit minimum distances, and the weights of the Boids plugin.
SEPARATION, ALIGNMENT, COHESION = FlockTerm(1.0, 5.0, -0.707, 12.0), FlockTerm(1.0, 7.5, 0.7, 8.0), FlockTerm(
    1.0, 9.0, -0.15, 8.0)
DT = 1.0 / 60.0


def listed():
    return [
        # One frame of the group flocking plugin at the Boids demo's size: the separate calls, then the agents
        # read back for drawing.  The smallest call: launches and latency.
        {"name": "frame-4k", "kind": "frame", "n": 4096, "radius": 50.0, "frames": 1, "mode": 1},
        # The same demo run as one call of 200 steps.
        {"name": "flock-4k", "kind": "flock", "n": 4096, "k": 7, "cells": "16,16,16", "size": 100.0, "wrap": "sphere",
         "steps": 200, "mode": 0, "on": "host"},
        # The group plugin's own default of 100,000 agents, an odd count, frame by frame with separate calls.
        {"name": "frames-100k", "kind": "frame", "n": 100003, "radius": 145.0, "frames": 60, "mode": 1},
        # A large flock, k = 7: the benchmark's state and lattice.
        {"name": "flock-1m-k7", "kind": "flock", "n": 1 << 20, "k": 7, "cells": "64,64,128", "size": 1000.0,
         "wrap": "box", "steps": 400, "mode": 0, "on": "device"},
        # The same flock with wide neighbourhoods, k = 16, on the lattice picked for it.
        {"name": "flock-1m-k16", "kind": "flock", "n": 1 << 20, "k": 16, "cells": "48,48,144", "size": 1000.0,
         "wrap": "box", "steps": 200, "mode": 0, "on": "device"},
        # The 10,000-agent choke-point crowd (two groups, walls, obstacles), frames issued by the library.
        {"name": "crowd-10k", "kind": "crowd", "n": 10000, "gap": 15.0, "frames": 100, "mode": 0},
        # The choke-point plugin on its parameter file: split walls, path, separate calls.
        {"name": "choke-131k", "kind": "choke", "n": 131072, "frames": 60, "walls": False},
        # The multi-group plugin on its parameter file: two groups avoiding each other.
        {"name": "groups-10k", "kind": "groups", "n": 5000, "frames": 40},
        # A parameter sweep: flocks and crowds of uneven size stepped together.
        {"name": "sweep-24", "kind": "ensemble", "scenarios": 24, "n_min": 1024, "n_max": 32768, "steps": 400},
        # One step of calibrating a crowd model: loss and gradient of a trajectory.
        {"name": "calibrate-16x8k", "kind": "calibrate", "scenarios": 16, "n": 8192, "steps": 50, "every": 10},
        # Brute-force search of a group in itself, lists read back.
        {"name": "brute-16k", "kind": "brute", "n": 16384, "m": 0, "k": 7},
        # Search among points that another program keeps on the device, at the entry point's largest size.
        {"name": "points-65k", "kind": "points", "n": 65536, "k": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "flock", "flock", "crowd", "choke", "groups", "ensemble", "calibrate", "brute",
                       "points"])
    if kind == "frame":
        n = _log(rng, 300, 100000)
        # the demo's density, from one frame with its read back to a run of frames
        return {"kind": kind, "n": n, "radius": round(50.0 * (n / 4096.0) ** (1.0 / 3.0), 3),
                "frames": rng.choice([1, 1, rng.randint(2, 60)]), "mode": rng.choice([0, 1])}
    if kind == "flock":
        n, k = _log(rng, 500, 1 << 20), rng.choice([4, 7, 7, 7, 8, 12, 16])
        wrap = rng.choice(["sphere", "box"]) if n < 200000 else "box"
        size = (1000.0 if wrap == "box" else 626.0) * (n / float(1 << 20)) ** (1.0 / 3.0)
        f = (n / float(1 << 20)) ** (1.0 / 3.0)
        base = rng.choice([(64, 64, 64), (64, 64, 128), (64, 64, 192)] if k <= 8 else [(48, 48, 96), (48, 48, 144)])
        cells = ",".join(str(max(4, int(round(c * f)))) for c in base)
        return {"kind": kind, "n": n, "k": k, "cells": cells, "size": round(size, 3), "wrap": wrap,
                "steps": rng.randint(20, 200), "mode": rng.choice([0, 0, 1]), "on": "device" if n > 30000 else "host"}
    if kind == "crowd":
        return {"kind": kind, "n": 2 * _log(rng, 300, 8000), "gap": rng.choice([7.5, 10.0, 15.0, 22.5, 30.0]),
                "frames": rng.randint(20, 100), "mode": rng.choice([0, 1])}
    if kind == "choke":
        return {"kind": kind, "n": _log(rng, 3000, 131072), "frames": rng.randint(10, 60),
                "walls": rng.choice([False, True])}
    if kind == "groups":
        return {"kind": kind, "n": _log(rng, 500, 5000), "frames": rng.randint(10, 40)}
    if kind == "ensemble":
        return {"kind": kind, "scenarios": rng.randint(3, 24), "n_min": 1024, "n_max": rng.choice([4096, 16384, 32768]),
                "steps": rng.randint(40, 300)}
    if kind == "calibrate":
        return {"kind": kind, "scenarios": rng.randint(1, 16), "n": 2 * _log(rng, 500, 4096),
                "steps": rng.randint(5, 50), "every": rng.choice([5, 10, 16])}
    if kind == "brute":
        n = _log(rng, 1000, 16384)
        return {"kind": kind, "n": n, "m": rng.choice([0, _log(rng, 300, 16384)]), "k": rng.choice([3, 7, 7, 10, 16])}
    return {"kind": kind, "n": _log(rng, 800, 65536), "k": rng.choice([4, 7, 8, 12, 16])}


# ---------------------------------------------------------------------------
# What a program holds before the pass.


class State(dict):
    """Handles and inputs of one program; the handles are closed with it."""

    def __del__(self):
        for h in self.get("close", ()):
            h.close()


_CTX = []


def _ctx():
    """The program's one context (device 0, its own stream)."""
    if not _CTX:
        _CTX.append(gs.Context(0))
    return _CTX[0]


def _rng(case, seed):
    return np.random.Generator(np.random.Philox(key=seed * 1000003 + int(case.get("n", 0))))


def _ball(g, n, radius):
    v = scenarios.unit_vectors(g, n) * (radius * g.uniform(0.0, 1.0, size=(n, 1)) ** (1.0 / 3.0))
    return v.astype(np.float32)


def _flock(g, pos):
    n = pos.shape[0]
    return scenarios.make_agents(pos, scenarios.unit_vectors(g, n), g.uniform(0.0, 9.0, size=n).astype(np.float32),
                                 0.5, 9.0, 27.0)


def _split_walls(params):
    return formats.WallSet.load_map(formats.DATA_DIR / params.map_filename).split(params.dimensions,
                                                                                params.cells).get()


def prepare(case, seed):
    ctx, g, kind = _ctx(), _rng(case, seed), case["kind"]
    s = State(case=dict(case), kind=kind)
    if kind == "frame":
        r = case["radius"]
        s["host"] = _flock(g, _ball(g, case["n"], r))
        s["radius"] = r
        s["group"] = gs.AgentGroup(ctx, s["host"])
        c = max(4, int(round(16 * (case["n"] / 4096.0) ** (1.0 / 3.0))))
        s["bins"] = gs.KNNBinData(ctx, (c, c, c), (2.2 * r,) * 3)
        s["knn"] = gs.KNNData(ctx, case["n"], 7)
        s["close"] = (s["knn"], s["bins"], s["group"])
    elif kind == "flock":
        n, size = case["n"], case["size"]
        cells = tuple(int(c) for c in case["cells"].split(","))
        if case["wrap"] == "box":
            pos = g.uniform(0.0, size, size=(n, 3)).astype(np.float32)
            p = scenarios.BoidsParams(k=case["k"], wrap_shape=0, wrap_center=(size / 2,) * 3, wrap_size=(size,) * 3,
                                      grid_origin=(0.0,) * 3, grid_size=(size,) * 3, grid_cells=cells)
        else:
            r = size / 2
            pos = _ball(g, n, r)
            p = scenarios.BoidsParams(k=case["k"], wrap_shape=1, wrap_center=(0.0,) * 3, wrap_size=(r, 0.0, 0.0),
                                      grid_origin=(-1.1 * r,) * 3, grid_size=(2.2 * r,) * 3, grid_cells=cells)
        p.mode = case["mode"]
        if p.mode == 1:
            p.separation, p.alignment, p.cohesion = SEPARATION, ALIGNMENT, COHESION
        s["host"], s["params"] = _flock(g, pos), p
        s["group"] = gs.AgentGroup(ctx, s["host"])
        s["bins"] = gs.KNNBinData(ctx, p.grid_cells, p.grid_size, origin=p.grid_origin)
        s["knn"] = gs.KNNData(ctx, n, p.k)
        s["close"] = (s["knn"], s["bins"], s["group"])
    elif kind == "crowd":
        # the plugin's 40 x 40 regions at their density of 3.1 agents per unit area
        region = 40.0 * math.sqrt(case["n"] / 10000.0)
        sc = scenarios.choke(n_total=case["n"], gap=case["gap"], workload=int(seed) % (1 << 40), region=region)
        sc.mode = case["mode"]
        if sc.mode == 1:
            sc.sep = FlockTerm(1.5, 3.0, -0.707, 10.0, 4096)
        s["sc"] = sc
        s["bins"] = gs.KNNBinData(ctx, sc.grid_cells, sc.grid_size, origin=sc.grid_origin)
        s["groups"] = [gs.AgentGroup(ctx, st) for st in sc.groups]
        s["walls"], s["obstacles"] = gs.WallGroup(ctx, sc.walls), gs.ObstacleGroup(ctx, *sc.obstacles)
        gs.updateKNNDatabase(s["walls"], s["bins"])
        gs.updateKNNDatabase(s["obstacles"], s["bins"])
        s["knns"] = [[gs.KNNData(ctx, st.n, k) for k in (sc.k, sc.k, sc.knw, sc.kno)] for st in sc.groups]
        s["close"] = [x for ks in s["knns"] for x in ks] + s["groups"] + [s["walls"], s["obstacles"], s["bins"]]
    elif kind == "choke":
        params = formats.load_params(formats.DATA_DIR / "ChokePoint.params")
        walls, mid = _split_walls(params)
        n = case["n"]
        sc = scenarios.choke_point_new(params, walls, mid, n_agents=16, dt=1.0 / 30.0)
        # a disc around the group's start that ends short of the wall, one agent to a half-unit square
        gp, radius = params.groups[0], 450.0 * math.sqrt(n / 131072.0)
        pos = np.zeros((0, 2), np.float32)
        while pos.shape[0] < n:
            rr, th = radius * np.sqrt(g.uniform(0.0, 1.0, 2 * n)), g.uniform(0.0, 2.0 * np.pi, 2 * n)
            pos = np.concatenate([pos, np.stack([rr * np.cos(th), 20.0 + radius + rr * np.sin(th)], 1).astype(np.float32)])
            _, first = np.unique(np.floor(pos / 0.5).astype(np.int64) @ np.array([1 << 20, 1]), return_index=True)
            pos = pos[np.sort(first)]
        pos = np.stack([pos[:n, 0], np.zeros(n, np.float32), pos[:n, 1]], 1)
        hd = g.uniform(0.0, 2.0 * np.pi, size=n)
        st = scenarios.make_agents(pos, np.stack([np.cos(hd), np.zeros(n), np.sin(hd)], 1), np.zeros(n, np.float32),
                                   0.5, gp.max_speed, gp.max_force)
        s["plugin"] = ChokePointNew(ctx, dataclasses.replace(sc, state=st))
        s["host"], s["group"] = st, s["plugin"].group
        s["close"] = (s["plugin"],)
    elif kind == "groups":
        params = formats.load_params(formats.DATA_DIR / "MultiGroup.params")
        sc = scenarios.multi_group(params, n_per_group=case["n"], dt=1.0 / 30.0, workload=int(seed) % (1 << 40))
        s["plugin"] = MultiGroup(ctx, sc)
        s["close"] = (s["plugin"],)
    elif kind == "ensemble":
        specs = _mix(case, int(seed))
        s["ens"] = Ensemble(ctx, specs)
        s["states"] = [(i, gi, st) for i, sp in enumerate(specs)
                       for gi, st in enumerate([sp[1]] if sp[0] == "boids" else sp[1].groups)]
        s["close"] = (s["ens"],)
    elif kind == "calibrate":
        specs = scenarios.calib_scenarios(case["scenarios"], case["n"], workload=int(seed) % (1 << 30))
        s["ens"] = Ensemble(ctx, specs)
        s["cal"] = Calibration(s["ens"], scenarios.CalibConfig(steps=case["steps"], checkpoint_every=case["every"]))
        s["theta"] = scenarios.calib_params() * g.uniform(0.8, 1.2, size=14)
        s["close"] = (s["cal"], s["ens"])
    elif kind == "brute":
        a = _flock(g, _ball(g, case["n"], 50.0))
        s["group"] = gs.AgentGroup(ctx, a)
        s["other"] = gs.AgentGroup(ctx, _flock(g, _ball(g, case["m"], 50.0))) if case["m"] else s["group"]
        s["knn"] = gs.KNNData(ctx, case["n"], case["k"])
        s["close"] = (s["knn"], s["group"]) + ((s["other"],) if case["m"] else ())
    elif kind == "points":
        n, k = case["n"], case["k"]
        s["pos"] = [torch.from_numpy(np.ascontiguousarray(c)).cuda() for c in _points(g, n).T]
        c = max(2, int((n / 2.0) ** (1.0 / 3.0)))
        s["bins"] = gs.KNNBinData(ctx, (c, c, c), (100.0,) * 3)
        s["idx"] = torch.empty((k, n), dtype=torch.int32, device="cuda")
        s["dist"] = torch.empty((k, n), dtype=torch.float32, device="cuda")
        s["close"] = (s["bins"],)
    return s


def _mix(case, seed):
    """Flocks and choke-point crowds in turn, of the sizes, weights and gaps of a sweep (the same for every seed)."""
    g, specs = scenarios.rng(3), []
    for i in range(case["scenarios"]):
        n = int(round(math.exp(g.uniform(math.log(case["n_min"]), math.log(case["n_max"])))))
        weights = g.uniform(0.7, 1.3, size=3)
        if i % 2 == 0:
            st, p = scenarios.boids_sphere(n=n, workload=seed * 1000 + i)
            for t, w in zip((p.separation, p.alignment, p.cohesion), weights):
                t.weight *= float(w)
            p.grid_cells = (scenarios.boids_cells_for(n, cell_factor=1.25),) * 3
            specs.append(("boids", st, p))
        else:
            n += n % 2
            sc = scenarios.choke(n_total=n, gap=7.5 + 2.5 * (i // 2 % 11), workload=seed * 1000 + i)
            c = scenarios.choke_cells_for(n, cell_factor=1.25)
            sc.grid_cells = (c, 1, c)
            specs.append(("choke", sc))
    return specs


def _points(g, n):
    """Half of the points spread over the box, half in a few loose clumps."""
    a = g.uniform(-50.0, 50.0, size=(n - n // 2, 3))
    c = g.uniform(-40.0, 40.0, size=(8, 3))[g.integers(0, 8, size=n // 2)] + 6.0 * g.normal(size=(n // 2, 3))
    return np.concatenate([a, c]).astype(np.float32)[g.permutation(n)]


# ---------------------------------------------------------------------------
# The pass.


class _View:
    def __init__(self, ptr, n, kind):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 2}


def _device_state(s):
    """The group's arrays where they are, in storage order, with the agent index of each slot.  Each tensor keeps
    the program's handles: the memory is the group's."""
    group, n = s["group"], s["case"]["n"]
    d = group.device_arrays()
    ids = ctypes.POINTER(ctypes.c_uint32)()
    capi.check(capi.lib.gs_group_device_order(group.h, ctypes.byref(ids), None), "gs_group_device_order")
    d["agent"] = ctypes.cast(ids, ctypes.c_void_p).value
    out = {}
    for f, ptr in d.items():
        out[f] = torch.as_tensor(_View(ptr, n, "<f4" if f in AGENT_FIELDS else "<i4"), device="cuda")
        out[f].owner = s
    return out


def _host_state(group):
    st = group.download()
    return dict(st.arrays, bits=st.bits)


def _frame(s):
    """The per-frame calls of the group flocking plugin."""
    A, knn, bins, mode = s["group"], s["knn"], s["bins"], s["case"]["mode"]
    gs.wrapWorld(A, shape=capi.GS_WRAP_SPHERE, radius=s["radius"])
    gs.updateKNNDatabase(A, bins)
    gs.findKNearestNeighbors(A, knn, bins, A, 1)
    for steer, t in ((gs.steerForSeparation, SEPARATION), (gs.steerForCohesion, COHESION),
                     (gs.steerForAlignment, ALIGNMENT)):
        steer(A, knn, A, t.min_d, t.max_d, t.cos_max, t.weight, t.mask, mode)
    gs.updateGroup(A, DT, mode)


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "frame":
        if case["frames"] == 1:  # an interactive program: the simulation goes on, and every frame is drawn
            _frame(s)
            return _host_state(s["group"])
        s["group"].upload(s["host"])
        for _ in range(case["frames"]):
            _frame(s)
        return _device_state(s)
    if kind == "flock":
        s["group"].upload(s["host"])
        api.stepBoids(s["group"], s["knn"], s["bins"], s["params"], case["steps"])
        return _host_state(s["group"]) if case["on"] == "host" else _device_state(s)
    if kind == "crowd":
        for G, st in zip(s["groups"], s["sc"].groups):
            G.upload(st)
        step_choke(s["groups"], s["knns"], s["walls"], s["obstacles"], s["bins"], s["sc"], case["frames"])
        return [_host_state(G) for G in s["groups"]]
    if kind == "choke":
        s["group"].upload(s["host"])
        (s["plugin"].step_with_wall_update if case["walls"] else s["plugin"].step)(case["frames"])
        return _device_state(s)
    if kind == "groups":
        for G, st in zip(s["plugin"].groups, s["plugin"].sc.states):
            G.upload(st)
        s["plugin"].step(case["frames"])
        return [_host_state(G) for G in s["plugin"].groups]
    if kind == "ensemble":
        for i, gi, st in s["states"]:
            s["ens"].upload(i, gi, st)
        s["ens"].step(case["steps"])
        got = [s["ens"].download(i, gi) for i, gi, _ in s["states"]]
        return {f: np.concatenate([st[f] for st in got]) for f in AGENT_FIELDS + ("bits",)}
    if kind == "calibrate":
        return {"loss": s["cal"].forward(s["theta"]), "grad": s["cal"].backward()}
    if kind == "brute":
        gs.findKNearestNeighborsBruteForce(s["group"], s["knn"], s["other"])
        idx, dist = s["knn"].download()
        return {"idx": idx, "dist": dist}
    p = [t.data_ptr() for t in s["pos"]]
    capi.check(capi.lib.gs_find_knn_noalloc(_ctx().h, s["bins"].h, case["n"], *p, case["k"], s["idx"].data_ptr(),
                                            s["dist"].data_ptr()), "gs_find_knn_noalloc")
    return {"idx": s["idx"], "dist": s["dist"]}


# ---------------------------------------------------------------------------
# What a pass cannot do without.


def _agents(case):
    if case["kind"] == "groups":
        return 2 * case["n"]
    if case["kind"] == "calibrate":
        return case["n"] * case["scenarios"]
    if case["kind"] == "ensemble":  # log-uniform sizes
        lo, hi = case["n_min"], case["n_max"]
        return int(case["scenarios"] * (hi - lo) / math.log(hi / lo))
    return case["n"]


def work(case):
    kind, n = case["kind"], _agents(case)
    if kind == "brute":
        m = case["m"] or n
        return {"bytes": 12.0 * n + (12.0 * m if case["m"] else 0.0) + 8.0 * case["k"] * n, "flops": 8.0 * n * m}
    if kind == "points":
        return {"bytes": (12.0 + 8.0 * case["k"]) * n, "flops": 8.0 * case["k"] * n}
    steps, k = case.get("steps", case.get("frames", 1)), case.get("k", 7)
    # Per agent and step: position, forward, speed, side and up read and written (104 bytes); k distances (8
    # operations each), three terms of about 10 a neighbour, and about 100 to integrate.  The walls, obstacles and
    # second group of a crowd add about as much again; a gradient needs every step forward twice and back once.
    flops = 38.0 * k + 100.0
    if kind in ("crowd", "choke", "groups", "calibrate"):
        flops *= 2.0
    passes = 3.0 if kind == "calibrate" else 1.0
    moved = 104.0 * n * steps * passes
    if kind != "calibrate":  # uploaded, and read back where that is part of the pass
        moved += 96.0 * n * 2
    return {"bytes": moved, "flops": flops * n * steps * passes}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits, for the passes that are one evaluation.  Rollouts have no such value: a flock or crowd is
# chaotic, and runs in 32 and in 64 bits part after some tens of steps.


def _nearest(a, b, k, same):
    """(index, distance) of the k nearest of b for each row of a, in 64 bits."""
    idx, dist = [], []
    for i in range(0, a.shape[0], 4096):
        q = a[i:i + 4096]
        d2 = sum((q[:, c, None] - b[None, :, c]) ** 2 for c in range(3))
        if same:
            r = torch.arange(q.shape[0], device=q.device)
            d2[r, r + i] = math.inf
        v, j = torch.topk(d2, k, dim=1, largest=False, sorted=True)
        idx.append(j)
        dist.append(v.sqrt())
    return torch.cat(idx), torch.cat(dist)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _norm(v):
    n = _dot(v, v).sqrt()
    return torch.where(n > 0, v / torch.where(n > 0, n, torch.ones_like(n)), v)


def _truncated(v, m):
    n = _dot(v, v).sqrt()
    return torch.where(n > m, v * (m / n.clamp_min(1e-300)), v)


def exact(case, seed):
    kind, g = case["kind"], _rng(case, seed)
    if kind == "points":
        p = torch.from_numpy(_points(g, case["n"])).cuda().double()
        return {"idx": None, "dist": _nearest(p, p, case["k"], True)[1].T.contiguous()}
    if kind == "brute":
        a = _flock(g, _ball(g, case["n"], 50.0))
        b = _flock(g, _ball(g, case["m"], 50.0)) if case["m"] else a
        p, q = (torch.from_numpy(x.pos()).cuda().double() for x in (a, b))
        return {"idx": None, "dist": _nearest(p, q, case["k"], not case["m"])[1].T.contiguous()}
    if kind != "frame" or case["frames"] != 1 or case["mode"] != 1:
        return None
    # one frame of the group plugin, by the formulas of the group kernels
    st = _flock(g, _ball(g, case["n"], case["radius"]))

    def of(x, y, z):
        return torch.from_numpy(np.stack([st[x], st[y], st[z]], 1)).cuda().double()

    pos, fwd, up, side = of("px", "py", "pz"), of("fx", "fy", "fz"), of("ux", "uy", "uz"), of("sx", "sy", "sz")
    speed = torch.from_numpy(st["speed"]).cuda().double()[:, None]
    r = _dot(pos, pos).sqrt()
    pos = torch.where(r > case["radius"], pos - 2 * case["radius"] * pos / r, pos)
    j, _ = _nearest(pos, pos, 7, True)
    off = pos[j] - pos[:, None]
    d2 = _dot(off, off)
    d = d2.sqrt()
    cone = _dot(fwd[:, None], off / d)
    steer = torch.zeros_like(pos)
    for t, v, rel in ((SEPARATION, -off / d2, torch.zeros_like(pos)), (COHESION, pos[j], pos), (ALIGNMENT, fwd[j], fwd)):
        near = (d < t.min_d) | ((d <= t.max_d) & (cone > t.cos_max))
        m = near.sum(1)
        mean = (v * near).sum(1) / m.clamp_min(1) - rel
        steer = steer + torch.where(m > 0, _norm(mean), torch.zeros_like(mean)) * t.weight
    vel = _truncated(fwd * speed + _truncated(steer, 27.0) * DT, 9.0)
    speed = _dot(vel, vel).sqrt()
    moving = speed > 0
    fwd = torch.where(moving, _norm(vel), fwd)
    side2 = _norm(torch.linalg.cross(fwd, up))
    side, up = torch.where(moving, side2, side), torch.where(moving, torch.linalg.cross(side2, fwd), up)
    pos = pos + vel * DT
    out = {f: torch.from_numpy(st[f].astype(np.float64)) for f in AGENT_FIELDS}
    for names, v in ((("px", "py", "pz"), pos), (("fx", "fy", "fz"), fwd), (("sx", "sy", "sz"), side),
                     (("ux", "uy", "uz"), up)):
        for c, f in enumerate(names):
            out[f] = v[:, c].contiguous()
    out["speed"] = speed[:, 0].contiguous()
    return dict(out, bits=None)

"""What a user of the engine has it do, as cases to time and to compare.

Every case goes through the public Python mirror of the C ABI (``cellflow_amd``) and covers
one way in which the engine is used:

* ``frame``    one widget frame: a step (with or without the proximity graph), then the
               particle records and the graph's line vertices to host memory.  The state
               advances from frame to frame.
* ``job``      a headless job: load a state, run a number of steps, read the state (and the
               graph) back.
* ``ensemble`` a batch of independent simulations advanced together, then read back.
* ``gradient`` one iteration of a fit: load the start state, roll out, gradient of the
               histogram loss with respect to the force table and the ratio.
* ``overlay``  what a renderer draws on a state that stands still: the proximity graph, its
               line vertices, the triangle mesh and its vertices.

Two physics: ``unit`` is that of the package's own workload files (boxes of a few units,
12,500 particles per unit volume, interaction radius 0.03 to 0.06, softness 1, dt 0.01);
``widget`` is that of the reference's preset files (20,000 to 30,000 particles spawned in
the central 2000^3 of an 8000^3 canvas, radius around 400), where every particle has
hundreds of neighbours.

``tuned`` cases set the tuning that the autotuner picks for the workload, as a program does
that keeps a tuning cache; the others run as the engine comes.
"""

import math

import numpy as np
import torch

from cellflow_amd import Ensemble, ParticleSimulation, SimulationParams, particles_from_state

# what cf_autotune picks: the 100k workload, the clustered one, the ensemble
TUNED = {
    "list": dict(cell_divisor=1, force_variant=4, lanes_per_particle=8, sort_variant=1),
    "dense": dict(cell_divisor=1, force_variant=0, lanes_per_particle=16, sort_variant=0),
    "batch": dict(cell_divisor=1, force_variant=3, lanes_per_particle=4, sort_variant=0),
}
DENSITY = 12500.0   # particles per unit volume of the package's uniform workloads
EDGE_CAP = 16       # connections per particle, the workloads' cap
MESH_ROOM = 8       # triangles per particle that an overlay's buffers hold
BINS, R_MAX = 32, 0.1


def listed():
    return [
        # the smallest call anyone makes in a loop: a toy frame, all launches and latency
        dict(name="frame_1k", kind="frame", physics="unit", n=1000, types=4, radius=0.05,
             ratio=0.3, balance=0.79, blobs=0, edges=0.02, tuned=""),
        # the widget as shipped: 20,000 particles of a preset, dense in the spawn cube
        dict(name="frame_preset_20k", kind="frame", physics="widget", n=20000, types=6,
             radius=397.0, ratio=0.0, balance=0.79, blobs=0, edges=60.0, tuned=""),
        # the widget with many particles: the readbacks of a frame are 8 MB
        dict(name="frame_100k", kind="frame", physics="unit", n=100000, types=8, radius=0.04,
             ratio=0.3, balance=0.79, blobs=0, edges=0.02, tuned=""),
        # the plain 10k workload, all its 100 steps
        dict(name="job_10k", kind="job", physics="unit", n=10000, types=6, radius=0.05,
             ratio=0.3, balance=0.79, blobs=0, edges=0.0, steps=100, tuned=""),
        # an odd count, ten types, few steps between readbacks
        dict(name="job_37k_odd", kind="job", physics="unit", n=37123, types=10, radius=0.0437,
             ratio=0.45, balance=1.1, blobs=0, edges=0.017, steps=7, tuned=""),
        # the 100k workload with its graph, as the engine comes
        dict(name="job_100k", kind="job", physics="unit", n=100000, types=8, radius=0.04,
             ratio=0.3, balance=0.79, blobs=0, edges=0.02, steps=100, tuned=""),
        # the same with the tuning of a program that autotunes
        dict(name="job_100k_tuned", kind="job", physics="unit", n=100000, types=8, radius=0.04,
             ratio=0.3, balance=0.79, blobs=0, edges=0.02, steps=100, tuned="list"),
        # half a million particles, no graph, as the engine comes
        dict(name="job_500k", kind="job", physics="unit", n=500009, types=8, radius=0.04,
             ratio=0.3, balance=0.79, blobs=0, edges=0.0, steps=50, tuned=""),
        # the clustered 1M workload's first steps, tuned: hundreds of neighbours each
        dict(name="job_1m_clustered", kind="job", physics="unit", n=1000000, types=8,
             radius=0.04, ratio=0.5, balance=1.2, blobs=200, edges=0.02, steps=20,
             tuned="dense"),
        # a quarter of the 256-member ensemble workload, tuned
        dict(name="ensemble_60", kind="ensemble", physics="unit", members=60, steps=200,
             tuned="batch"),
        # the differentiable 20k rollout, all its 200 steps
        dict(name="gradient_20k", kind="gradient", physics="unit", n=20000, types=6,
             radius=0.05, ratio=0.3, balance=0.79, blobs=0, steps=200, every=20, tuned=""),
        # both overlays of a clumped state
        dict(name="overlay_50k", kind="overlay", physics="unit", n=50000, types=4, radius=0.04,
             ratio=0.3, balance=0.79, blobs=800, edges=0.02, tuned=""),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "job", "job", "job", "clustered", "ensemble",
                       "gradient", "overlay"])
    if kind == "ensemble":
        return dict(kind=kind, physics="unit", members=_log(rng, 3, 60),
                    steps=rng.randint(50, 200), tuned=rng.choice(["", "batch"]))
    base = dict(types=rng.randint(2, 10), radius=round(rng.uniform(0.03, 0.06), 5),
                ratio=round(rng.uniform(0.0, 0.5), 3), balance=round(rng.uniform(0.6, 1.3), 3),
                blobs=0)
    if kind == "frame" and rng.random() < 0.4:
        base.update(radius=round(rng.uniform(280.0, 630.0), 1), ratio=0.0)
        return dict(kind=kind, physics="widget", n=_log(rng, 5000, 30000),
                    edges=rng.choice([0.0, round(rng.uniform(20.0, 100.0), 1)]), tuned="", **base)
    edges = rng.choice([0.0, round(rng.uniform(0.3, 0.6) * base["radius"], 5)])
    if kind == "frame":
        return dict(kind=kind, physics="unit", n=_log(rng, 500, 100000), edges=edges,
                    tuned=rng.choice(["", "", "list"]), **base)
    if kind == "clustered":
        n = _log(rng, 50000, 1000000)
        base.update(radius=round(rng.uniform(0.03, 0.04), 5),
                    blobs=max(10, n // rng.randint(1000, 5000)))
        edges = edges and round(rng.uniform(0.3, 0.6) * base["radius"], 5)
        return dict(kind="job", physics="unit", n=n, edges=edges, steps=rng.randint(5, 20),
                    tuned=rng.choice(["", "dense"]), **base)
    if kind == "job":
        n = _log(rng, 2000, 500000)
        return dict(kind=kind, physics="unit", n=n, edges=edges,
                    steps=min(rng.randint(5, 100), max(5, 20000000 // n)),
                    tuned=rng.choice(["", "", "list"]), **base)
    if kind == "gradient":
        base.update(types=rng.randint(2, 8), balance=0.79)
        return dict(kind=kind, physics="unit", n=_log(rng, 3000, 20000),
                    steps=rng.randint(40, 200), every=rng.randint(8, 24), tuned="", **base)
    n = _log(rng, 2000, 50000)
    base.update(radius=round(rng.uniform(0.03, 0.045), 5), types=rng.randint(4, 10),
                blobs=max(4, n // rng.randint(40, 70)))
    return dict(kind="overlay", physics="unit", n=n,
                edges=round(rng.uniform(0.3, 0.5) * base["radius"], 5), tuned="", **base)


# ---- inputs ------------------------------------------------------------------------------


def _start(case, seed):
    """Box, positions, types, force table and radius modifiers of a case, from the seed."""
    rng = np.random.default_rng([seed, case["n"], case["types"]])
    n, T = case["n"], case["types"]
    if case["physics"] == "widget":
        side = 8000.0
        pos = 3000.0 + 2000.0 * rng.random((n, 3))
        raw = rng.uniform(-1.0, 1.0, T * T).astype(np.float32)
        table = None
    else:
        density = DENSITY if not case["blobs"] else 4630.0
        side = float(np.float32((n / density) ** (1.0 / 3.0)))
        if case["blobs"]:
            # overlays: clumps with a few connections per particle; jobs: wide dense blobs
            sd = 0.02 if case["kind"] == "overlay" else 0.05
            centres = side * rng.random((case["blobs"], 3))
            pos = centres[rng.integers(0, case["blobs"], n)] + sd * rng.standard_normal((n, 3))
            pos = np.mod(pos, side)
        else:
            pos = side * rng.random((n, 3))
        table = rng.normal(0.1 if case["kind"] != "gradient" else 0.0,
                           0.6 if case["kind"] != "gradient" else 0.5, (T, T)).astype(np.float32)
        raw = None
    below = np.nextafter(np.float32(side), np.float32(0))
    pos = np.minimum(pos.astype(np.float32), below)
    ptype = rng.integers(0, T, n).astype(np.uint32)
    rbt = rng.uniform(-1.0, 1.0, T).astype(np.float32)
    return dict(side=side, pos=pos, type=ptype, table=table, raw=raw, rbt=rbt,
                colors=rng.random((T, 3)).astype(np.float32))


def _params(case, side):
    widget = case["physics"] == "widget"
    return SimulationParams(
        radius=case["radius"], delta_t=0.13 if widget else 0.001 if case["kind"] == "gradient"
        else 0.01, friction=0.44 if widget else 0.1, repulsion=162.7 if widget else 64.83,
        attraction=0.97 if widget else 3.06, k=27.93 if widget else 1.0, balance=case["balance"],
        canvasWidth=side, canvasHeight=side, canvasDepth=side, numParticleTypes=case["types"],
        ratioWithLFO=case["ratio"], forceMultiplier=2.33, maxExpectedNeighbors=400)


FORCE_RANGE, FORCE_BIAS, FORCE_OFFSET = 0.33, -0.185, 0.79  # a preset's updateForceTable


def _sizes(case):
    """Particle counts of an ensemble's members, log-uniform in 2,000 to 50,000."""
    rng = np.random.default_rng([case["members"], case["steps"]])
    u = rng.uniform(math.log(2000), math.log(50000), case["members"])
    return [int(n) for n in np.round(np.exp(u))]


def _members(case, seed):
    """The member simulations of an ensemble: uneven sizes, types, radii, own force tables."""
    rng = np.random.default_rng([seed, case["members"]])
    out = []
    for n in _sizes(case):
        T = int(rng.integers(4, 9))
        side = float(np.float32((n / DENSITY) ** (1.0 / 3.0)))
        pos = np.minimum((side * rng.random((n, 3))).astype(np.float32),
                         np.nextafter(np.float32(side), np.float32(0)))
        phys = dict(radius=float(rng.uniform(0.03, 0.06)), delta_t=0.01, friction=0.1,
                    repulsion=64.83, attraction=3.06, k=1.0, balance=0.79, canvas=[side] * 3,
                    num_types=T, ratio=0.3, force_multiplier=2.33, max_expected_neighbors=400)
        out.append((phys, dict(pos=pos, vel=np.zeros((n, 3), np.float32),
                               type=rng.integers(0, T, n).astype(np.uint32),
                               table=rng.normal(0.0, 0.5, (T, T)).astype(np.float32),
                               rbt=rng.uniform(-1.0, 1.0, T).astype(np.float32))))
    return out


def _target(side, n, seed):
    """A histogram to fit: an ideal gas's with random features."""
    w = R_MAX / BINS
    c = (np.arange(BINS) + 0.5) * w
    bumps = 1.0 + 0.3 * np.random.default_rng([seed, 7]).standard_normal(BINS)
    return n / side ** 3 * 4.0 * math.pi * c * c * w * bumps


def prepare(case, seed):
    if case["kind"] == "ensemble":
        ens = Ensemble(_members(case, seed))
        if case["tuned"]:
            ens.setTuning(**TUNED[case["tuned"]])
        return dict(case=case, ens=ens)
    st = _start(case, seed)
    sim = ParticleSimulation(case["n"], case["types"])
    if st["table"] is not None:
        sim.setForceTable(st["table"])
    else:
        sim.setRawForceTableValues(st["raw"])
        sim.updateForceTable(FORCE_RANGE, FORCE_BIAS, FORCE_OFFSET)
    sim.setRadioByType(st["rbt"])
    if case["tuned"]:
        sim.setTuning(**TUNED[case["tuned"]])
    zero = np.zeros_like(st["pos"])
    records = particles_from_state(st["pos"], zero, st["type"])
    params = _params(case, st["side"])
    s = dict(case=case, sim=sim, params=params, start=records, colors=st["colors"],
             out=np.empty_like(records))
    n = case["n"]
    if case["kind"] in ("frame", "overlay"):
        sim.setParticles(records)
        # a vertex buffer of the most a graph of this cap can hold, as a VBO is sized
        s["lines"] = np.zeros((2 * EDGE_CAP * n, 6), np.float32)
    if case["kind"] in ("job", "overlay"):
        s["edges"] = np.zeros((EDGE_CAP * n, 2), np.int32)
    if case["kind"] == "overlay":
        sim.simulate(params, 0)
        s["tris"] = np.zeros((MESH_ROOM * n, 3), np.int32)
        s["mesh"] = np.zeros((3 * MESH_ROOM * n, 9), np.float32)
    if case["kind"] == "gradient":
        s["target"] = _target(st["side"], n, seed)
    return s


# ---- one pass ----------------------------------------------------------------------------


def _fields(rec):
    return dict(pos=rec["pos"], vel=rec["vel"], acc=rec["acc"], ptype=rec["ptype"])


def _into(buffer, rows):
    """Rows at the head of the program's own buffer, and how many."""
    buffer[:len(rows)] = rows
    return dict(buffer=buffer, count=len(rows))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ensemble":
        s["ens"].simulate(case["steps"])
        # the 44-byte records of every member, as rows of 11 words
        return [s["ens"].getParticleData(m).view(np.float32).reshape(-1, 11)
                for m in range(case["members"])]
    sim, params = s["sim"], s["params"]
    if kind == "gradient":
        sim.setParticles(s["start"])
        loss, hist, table, ratio = sim.rolloutGrad(params, case["steps"], case["every"], BINS,
                                                   R_MAX, s["target"])
        return dict(loss=loss, hist=hist, table=table, ratio=ratio)
    if kind == "overlay":
        edges = _into(s["edges"], sim.generateProximityGraph(case["edges"], EDGE_CAP))
        sim.getLineVertices(s["colors"], out=s["lines"])
        tris = _into(s["tris"], sim.generateTriangleMesh(case["edges"], EDGE_CAP))
        sim.getTriangleVertices(s["colors"], out=s["mesh"])
        return dict(edges=edges, lines=s["lines"], tris=tris, mesh=s["mesh"])
    edges = (case["edges"], EDGE_CAP) if case["edges"] else None
    if kind == "frame":
        sim.simulate(params, 1, edges=edges)
        out = _fields(sim.getParticleData(out=s["out"]))
        if edges:
            out["count"] = len(sim.getLineVertices(s["colors"], out=s["lines"]))
            out["lines"] = s["lines"]
        return out
    sim.setParticles(s["start"])
    sim.simulate(params, case["steps"], edges=edges)
    out = _fields(sim.getParticleData(out=s["out"]))
    if edges:
        out["edges"] = _into(s["edges"], sim.getEdges())
    return out


# ---- what a pass cannot do without -------------------------------------------------------

STEP_BYTES = 60.0    # per particle and step: position, velocity, type, count in and out
PAIR_FLOPS = 25.0    # per in-range pair


def _neighbours(case):
    """In-range neighbours of a particle, from the density around it."""
    if case["physics"] == "widget":
        density = case["n"] / 2000.0 ** 3
    elif case["blobs"]:
        sd = 0.02 if case["kind"] == "overlay" else 0.05
        density = 4630.0 + case["n"] / case["blobs"] / (4.0 * math.pi * sd * sd) ** 1.5
    else:
        density = DENSITY
    return min(case["n"], density * 4.0 / 3.0 * math.pi * case["radius"] ** 3)


def work(case):
    if case["kind"] == "ensemble":
        n = float(sum(_sizes(case))) * case["steps"]
        # radius uniform in 0.03 to 0.06
        near = DENSITY * 4.0 / 3.0 * math.pi * 0.0456 ** 3
        return {"bytes": STEP_BYTES * n, "flops": PAIR_FLOPS * near * n}
    n, near = case["n"], _neighbours(case)
    if case["kind"] == "gradient":
        # a step forward and a step back, the state in FP64
        return {"bytes": 4.0 * STEP_BYTES * n * case["steps"],
                "flops": 4.0 * PAIR_FLOPS * near * n * case["steps"]}
    if case["kind"] == "overlay":
        near = near * (case["edges"] / case["radius"]) ** 3 / case["types"]
        edges = n * min(EDGE_CAP, near / 2.0)
        return {"bytes": 32.0 * n + (8.0 + 48.0 + 12.0 + 108.0) * edges,
                "flops": 10.0 * near * n}
    steps = case.get("steps", 1)
    return {"bytes": (STEP_BYTES + (20.0 if case["edges"] else 0.0)) * n * steps + 44.0 * n,
            "flops": PAIR_FLOPS * near * n * steps}


# ---- the same in 64 bits -----------------------------------------------------------------


def _f(x):
    """An FP32 parameter's value."""
    return float(np.float32(x))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _wrapped(d, side):
    """Differences shifted by one period where they exceed half a side."""
    d = torch.where(d > 0.5 * side, d - side, d)
    return torch.where(d < -0.5 * side, d + side, d)


def _within(x, reach, side, same=None):
    """Ordered pairs (i, j), i != j, nearer than `reach` (scalar, or by type pair through
    `same` = (reach table, types)); `side` None: no periodic images."""
    n = x.shape[0]
    rows = max(1, min(n, 40000000 // n))
    out = []
    for r0 in range(0, n, rows):
        xi = x[r0:r0 + rows]
        s = torch.zeros((xi.shape[0], n), dtype=x.dtype, device=x.device)
        for a in range(3):
            d = x[None, :, a] - xi[:, a, None]
            if side is not None:
                d = _wrapped(d, side)
            s += d * d
        if same is None:
            hit = s < reach * reach
        else:
            hit = torch.sqrt(s + _f(1e-4)) < same[0][same[1][r0:r0 + rows]][:, same[1]]
        hit[torch.arange(xi.shape[0], device=x.device), torch.arange(r0, r0 + xi.shape[0],
                                                                     device=x.device)] = False
        i, j = torch.nonzero(hit, as_tuple=True)
        out.append((i + r0, j))
    return torch.cat([p[0] for p in out]), torch.cat([p[1] for p in out])


def _step64(x, v, prev, t, p, side, table, ratio, rbt):
    """One step in 64 bits: new positions, velocities, counts, accelerations."""
    eff_t = _f(p.radius) * (1.0 + rbt * ratio)
    eff = 0.5 * (eff_t[:, None] + eff_t[None, :])
    with torch.no_grad():
        i, j = _within(x, None, side, (eff.detach(), t))
    d = _wrapped(x[j] - x[i], side)
    dist = torch.sqrt((d * d).sum(1) + _f(1e-4))
    rr = dist / eff[t[i], t[j]]
    net = (_f(p.repulsion) * torch.exp(-_f(p.k) * rr * rr) - _f(p.attraction) * rr) \
        * table[t[i], t[j]]
    f = torch.zeros_like(x).index_add(0, i, d / dist[:, None] * net[:, None])
    cnt = torch.bincount(i, minlength=x.shape[0])
    dens = torch.clamp((cnt + prev) * 0.5 / p.maxExpectedNeighbors, max=1.0)
    f = f * (_f(p.forceMultiplier) * (1.0 - (1.0 - _f(p.balance)) * dens))[:, None]
    v = v * _f(p.friction) + f * _f(p.delta_t)
    return torch.remainder(x + v * _f(p.delta_t), side), v, cnt, f


def _mesh64(pos, ptype, distance, colors):
    """Triangles of the mesh rule (same type, within 1.2 distances, non-periodic; the first
    EDGE_CAP neighbours by index; fans over those above the owner, at most 64) and their
    vertices' position, flat normal and colour."""
    x = torch.as_tensor(pos, device=_device()).double()
    i, j = (v.cpu().numpy() for v in _within(x, 1.2 * _f(distance), None))
    keep = ptype[i] == ptype[j]
    i, j = i[keep], j[keep]
    order = np.lexsort((j, i))
    i, j = i[order], j[order]
    first = np.searchsorted(i, np.arange(len(pos) + 1))
    tris = []
    for o in np.unique(i):
        near = j[first[o]:first[o + 1]][:EDGE_CAP]
        near = near[near > o]
        a, b = np.triu_indices(len(near), 1)
        tris.append(np.stack([np.full(len(a[:64]), o), near[a[:64]], near[b[:64]]], 1))
    tris = np.concatenate(tris) if tris else np.zeros((0, 3), np.int64)
    v = pos.astype(np.float64)[tris]
    normal = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    length = np.linalg.norm(normal, axis=1, keepdims=True)
    normal = np.where(length > _f(1e-4), normal / np.maximum(length, 1e-300), normal)
    col = colors.astype(np.float64)[ptype[tris[:, 0]]]
    rows = np.concatenate([v, np.repeat(normal[:, None], 3, 1), np.repeat(col[:, None], 3, 1)], 2)
    out = np.zeros((3 * MESH_ROOM * len(pos), 9))
    out[:3 * len(rows)] = rows.reshape(-1, 9)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "job"):
        # many steps of a chaotic system: the 64-bit trajectory from the same start is
        # another one after a few tens of steps
        return None
    st = _start(case, seed)
    if kind == "overlay":
        return dict(edges=None, lines=None, tris=None,
                    mesh=_mesh64(st["pos"], st["type"], case["edges"], st["colors"]))
    dev = _device()
    p = _params(case, st["side"])
    side = _f(st["side"])
    x = torch.as_tensor(st["pos"], device=dev).double()
    v = torch.zeros_like(x)
    t = torch.as_tensor(st["type"].astype(np.int64), device=dev)
    rbt = torch.as_tensor(st["rbt"], device=dev).double()
    if st["table"] is not None:
        table = torch.as_tensor(st["table"], device=dev).double()
    else:
        raw = torch.as_tensor(st["raw"], device=dev).double().reshape(case["types"], -1)
        table = torch.clamp(torch.tanh(raw * _f(FORCE_OFFSET)) * _f(FORCE_RANGE) + _f(FORCE_BIAS),
                            -1.0, 1.0)
    prev = torch.zeros(case["n"], dtype=torch.int64, device=dev)
    if kind == "frame":
        x, v, _, f = _step64(x, v, prev, t, p, side, table, _f(p.ratioWithLFO), rbt)
        out = dict(pos=x, vel=v, acc=f, ptype=None)
        return dict(out, count=None, lines=None) if case["edges"] else out
    # the gradient, by torch's autograd over the rollout
    table = table.requires_grad_()
    ratio = torch.tensor(_f(p.ratioWithLFO), dtype=torch.float64, device=dev, requires_grad=True)
    for _ in range(case["steps"]):
        x, v, prev, _ = _step64(x, v, prev, t, p, side, table, ratio, rbt)
    w = R_MAX / BINS
    with torch.no_grad():
        i, j = _within(x, R_MAX + 2.0 * w, side)
    u = torch.sqrt((_wrapped(x[j] - x[i], side) ** 2).sum(1)) / w - 0.5
    hist = []
    for b in range(BINS):
        a = torch.abs(u - b)
        near = (4.0 - 6.0 * a * a + 3.0 * a ** 3) / 6.0
        far = torch.clamp(2.0 - a, min=0.0) ** 3 / 6.0
        hist.append(torch.where(a < 1.0, near, far).sum() / case["n"])
    hist = torch.stack(hist)
    target = torch.as_tensor(_target(st["side"], case["n"], seed), device=dev)
    loss = ((hist - target) ** 2).sum()
    loss.backward()
    return dict(loss=float(loss.detach()), hist=hist.detach(), table=table.grad,
                ratio=float(ratio.grad))

"""Performance cases of the library: what its users have it do, through its
public entry points (capi.Context and the C ABI below it).

listed() holds one case per use, draw() makes more of the same ranges.  A case
is a dict of plain values whose "kind" is one of

  sheet   one cloth, one frame of 10 substeps (Gauss-Seidel projection of
          distance, and with bend of dihedral prims), state read back
  scenes  many 32 x 32 cloths with wind, pins and a sphere in one context,
          one frame, state read back
  batch   many cloths of uneven size in one context, one frame, state read
          back; warm: with the learned warm start and its fallback
  drape   a cloth falling onto a static icosphere with continuous collision
          detection, one frame
  fold    a folded cloth over a static box with self contact, one frame
  detect  standalone contact detection and response on host arrays
  hash    spatial-hash build on device arrays, no allocation
  train   one epoch of the warm-start network

Every frame starts from a device snapshot of the prepared state (as a rollout
from a stored state does), so that each pass does the same work.
"""
import ctypes as C
import math

import numpy as np
import torch

from positionbaseddynamicsold_amd import capi, scenes

DT = 1.0 / 600.0
SUBSTEPS = 10


def listed():
    return [
        # the smallest scene a user steps: one 32 x 32 cloth hung by two corners, default settings
        dict(name="sheet_32", kind="sheet", rx=32, ry=32, bend=False, sphere=False, iterations=20, graph=0,
             tile_sweeps=0, tile_max_verts=0),
        # one garment-sized cloth of odd sides, default settings
        dict(name="sheet_389x211", kind="sheet", rx=389, ry=211, bend=False, sphere=False, iterations=20, graph=0,
             tile_sweeps=0, tile_max_verts=0),
        # a fine cloth with bending over an analytic sphere, graph replay
        dict(name="sheet_bend_256", kind="sheet", rx=256, ry=256, bend=True, sphere=True, iterations=20, graph=1,
             tile_sweeps=2, tile_max_verts=5104),
        # many small scenes side by side: data generation, rollouts
        dict(name="scenes_256", kind="scenes", count=256, iterations=20, graph=1),
        # cloths of uneven size in one context at the launch shape the autotuner picks for such batches: the plain
        # solver, and the warm start with its per-cloth fallback
        dict(name="batch_48", kind="batch", count=48, layout=0, warm=False, iterations=20, graph=1, tile_sweeps=2,
             tile_max_verts=5104),
        dict(name="batch_48_warm", kind="batch", count=48, layout=0, warm=True, iterations=20, graph=1, tile_sweeps=2,
             tile_max_verts=0),
        # cloth against a static mesh: bending, swept-box candidates
        dict(name="drape_128", kind="drape", n=128, robust=True, edge_edge=False, iterations=20),
        # self contact with the reference's centroid-cell candidates
        dict(name="fold_256", kind="fold", n=256, robust=False, edge_edge=False, iterations=30),
        # self contact with edge-edge contacts beside the vertex-face ones
        dict(name="fold_ee_96", kind="fold", n=96, robust=True, edge_edge=True, iterations=30),
        # a caller with its own integrator that only wants contacts found and resolved
        dict(name="detect_96", kind="detect", n=96, swept=False),
        # the broadphase table of a large mesh, built in place on the caller's stream
        dict(name="hash_512", kind="hash", n=512, mode=1, table_bits=22),
        # one epoch of training the warm-start network on collected samples
        dict(name="train_64k", kind="train", samples=65536, batch=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sheet", "sheet", "sheet", "scenes", "batch", "batch", "drape", "fold", "fold", "detect",
                       "hash", "hash", "train"])
    if kind == "sheet":
        bend = rng.random() < 0.35
        top = 256 if bend else 512
        tuned = rng.random() < 0.5
        return dict(kind=kind, rx=_log_int(rng, 16, top), ry=_log_int(rng, 16, top), bend=bend,
                    sphere=rng.random() < 0.5, iterations=rng.randint(8, 24), graph=rng.randint(0, 1),
                    tile_sweeps=2 if tuned else 0, tile_max_verts=5104 if tuned else 0)
    if kind == "scenes":
        return dict(kind=kind, count=_log_int(rng, 16, 500), iterations=rng.randint(8, 24), graph=rng.randint(0, 1))
    if kind == "batch":
        warm = rng.random() < 0.4
        return dict(kind=kind, count=_log_int(rng, 6, 64), layout=rng.randint(1, 10 ** 6), warm=warm, iterations=rng.randint(16, 22), graph=1,
                    tile_sweeps=2, tile_max_verts=0 if warm else 5104)
    if kind == "drape":
        return dict(kind=kind, n=_log_int(rng, 40, 140), robust=rng.random() < 0.7, edge_edge=False,
                    iterations=rng.randint(10, 20))
    if kind == "fold":
        ee = rng.random() < 0.3
        return dict(kind=kind, n=_log_int(rng, 40, 90) if ee else _log_int(rng, 60, 240),
                    robust=ee or rng.random() < 0.5, edge_edge=ee, iterations=rng.randint(10, 28))
    if kind == "detect":
        return dict(kind=kind, n=_log_int(rng, 20, 130), swept=rng.random() < 0.5)
    if kind == "hash":
        dense = rng.random() < 0.3
        return dict(kind=kind, n=_log_int(rng, 24, 700), mode=0 if dense else 1,
                    table_bits=0 if dense else rng.randint(12, 22))
    return dict(kind=kind, samples=_log_int(rng, 6000, 100000), batch=rng.choice([1000, 2048, 4096, 6000]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _boundary(rx, ry):
    i = np.arange(rx * ry)
    return i[(i % rx == 0) | (i % rx == rx - 1) | (i < rx) | (i >= (ry - 1) * rx)]


def _specs(case, seed):
    """The cloths of a sheet, scenes or batch case, as plain numbers (a batch's sizes are its layout's)."""
    rng = np.random.default_rng([case.get("layout", seed), 77])
    f = lambda v: float(np.float32(v))  # noqa: E731
    out = []
    if case["kind"] == "sheet":
        rx, ry = case["rx"], case["ry"]
        sx, sy = 1.0, f((ry - 1) / (rx - 1))
        sphere = ((f(0.5 * sx), f(-0.302), f(0.5 * sy)), f(0.3)) if case["sphere"] else None
        out.append(dict(rx=rx, ry=ry, sx=sx, sy=sy, pins=[] if sphere else [0, rx - 1], sphere=sphere, wind=None))
    elif case["kind"] == "scenes":
        for _ in range(case["count"]):
            npins = int(rng.integers(0, 5))
            ang, speed = rng.uniform(0, 2 * np.pi), rng.uniform(0, 5)
            c = (f(rng.uniform(0.2, 0.8)), f(rng.uniform(-0.35, -0.29)), f(rng.uniform(0.2, 0.8)))
            out.append(dict(rx=32, ry=32, sx=1.0, sy=1.0, pins=sorted(rng.choice(_boundary(32, 32), npins, False).tolist()),
                            sphere=(c, f(0.3)), wind=(f(speed * np.cos(ang)), 0.0, f(speed * np.sin(ang)))))
    else:
        for _ in range(case["count"]):
            side, aspect = int(rng.integers(16, 257)), rng.uniform(0.5, 2.0)
            rx, ry = side, max(2, int(round(side * aspect)))
            npins = int(rng.integers(0, 5))
            r = f(rng.uniform(0.2, 0.4))
            out.append(dict(rx=rx, ry=ry, sx=1.0, sy=f(aspect), wind=None,
                            pins=sorted(rng.choice(_boundary(rx, ry), npins, False).tolist()),
                            sphere=((0.5, f(-r - 0.02), f(0.5 * aspect)), r)))
    for k, s in enumerate(out):
        s["jitter"], s["seed"] = 1e-4, int(seed) * 100003 + k
    return out


def _velocity(seed, n):
    """Start velocities: a common fall with some turbulence."""
    rng = np.random.default_rng([seed, 78])
    return (np.array([0.0, -0.5, 0.0]) + 0.05 * rng.standard_normal((n, 3))).astype(np.float32)


def _cloths(case, seed):
    ctx = capi.Context(0)
    bend = case.get("bend", False)
    for s in _specs(case, seed):
        c = ctx.add_grid(s["rx"], s["ry"], s["sx"], s["sy"], jitter=s["jitter"], seed=s["seed"])
        ctx.set_constraint_option(c, capi.DISTANCE | (capi.BENDING if bend else 0), (1.0, 0.1, 1.0))
        if s["pins"]:
            ctx.set_pins(c, s["pins"])
        kw = {}
        if s["sphere"]:
            kw.update(sphere_on=1, sphere_c=s["sphere"][0], sphere_r=s["sphere"][1])
        if s["wind"]:
            kw.update(wind=s["wind"], wind_drag=1.0)
        if kw:
            ctx.set_params(c, **kw)
    ctx.init()
    return ctx


def _moving(case, seed, kw):
    ctx = _cloths(case, seed)
    ctx.set_solver(**kw)
    x, _ = ctx.state_save()
    ctx.state_load(x, _velocity(seed, len(x)))
    return ctx


def _contact_scene(case, seed):
    if case["kind"] == "drape":
        sc = scenes.config2(n=case["n"], seed=seed % 1000003)
        sc.cloth.origin = (-0.5, 0.303, -0.5)
    else:
        sc = scenes.config3(n=case["n"], seed=seed % 1000003, box_div=max(8, case["n"] // 8))
        sc.cloth.origin = (-0.5, 0.403, -0.5)
    if case["robust"]:
        sc = sc.robust()
    sc.edge_edge = 1 if case["edge_edge"] else 0
    sc.iterations = case["iterations"]
    ctx = capi.Context(0)
    cloth, static, _ = scenes.add_ccd_scene(ctx, sc)
    v = _velocity(seed, ctx.info(cloth).nv)
    v[:, 1] -= 0.5
    ctx.set(cloth, capi.STATE_V, v)
    return ctx


def _grid_tris(n, m):
    i = (np.arange(m - 1)[:, None] * n + np.arange(n - 1)[None, :]).reshape(-1)
    return np.stack([i, i + n, i + n + 1, i, i + n + 1, i + 1], 1).reshape(-1, 3).astype(np.int32)


def _wavy_sheet(n, rng):
    g = np.arange(n) / (n - 1)
    x, z = np.tile(g, n), np.repeat(g, n)
    y = 0.05 * np.sin(6.0 * x + rng.uniform(0, 6)) * np.cos(5.0 * z) + 0.1 / n * rng.standard_normal(n * n)
    return np.stack([x, y, z], 1).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("sheet", "scenes", "batch"):
        kw = dict(dt=DT, iterations=case["iterations"], graph=case["graph"], tile_sweeps=case.get("tile_sweeps", 0),
                  tile_max_verts=case.get("tile_max_verts", 0))
        ctx = _moving(case, seed, kw)
        if case.get("warm"):
            # weights trained on samples the solver recorded on other cloths, both sets some substeps into their fall
            other = _moving(dict(case, count=16, layout=case["layout"] + 1), seed, kw)
            other.step(12)
            other.ws_init(seed % 1000)
            other.ws_collect(60, 1)
            other.ws_train(4, 4096, 1e-3, 0)
            ctx.ws_set_params(other.ws_params())
            ctx.ws_set_norm(other.ws_norm())
            other.close()
            ctx.step(12)
            ctx.set_solver(warm_iterations=1, warm_rule=1, warm_gate=1e-4, **kw)
            ctx.ws_enable(True)
        ctx.snapshot(False)
        return dict(kind="step", ctx=ctx)
    if kind in ("drape", "fold"):
        ctx = _contact_scene(case, seed)
        ctx.snapshot(False)
        return dict(kind="contact", ctx=ctx)
    rng = np.random.default_rng([seed, 79])
    if kind == "detect":
        # two layers of one folded sheet closing on each other over a step
        n = case["n"]
        h = 1.0 / (n - 1)
        x = _wavy_sheet(n, rng).astype(np.float64)
        flip = x[:, 0] > 0.5
        x[:, 1] *= 0.2
        x[flip, 0] = 1.0 - x[flip, 0]
        x[flip, 1] += 0.8 * h
        p = x + 0.02 * h * rng.standard_normal(x.shape)
        p[flip, 1] -= h * rng.uniform(0.2, 0.9, int(flip.sum()))
        # the caller's own contact arrays, filled from the front
        room = 16 * n * n
        got = [np.zeros((room, 2), np.int32), np.zeros(room, np.float32), np.zeros((room, 3), np.float32),
               np.zeros((room, 4), np.float64)]
        return dict(kind=kind, ctx=capi.Context(0), got=got, count=0, x=x.astype(np.float32), p=p.astype(np.float32),
                    tris=_grid_tris(n, n), w=np.ones(n * n, np.float32), th=0.1 * h, swept=case["swept"],
                    desc=capi.hash_desc(1, cell=(1.8 * h,) * 3, table_bits=18))
    if kind == "hash":
        n = case["n"]
        pos, tris = _wavy_sheet(n, rng), _grid_tris(n, n)
        cell = 1.5 * 1.14 / (n - 1)
        dims = tuple(min(400, int(math.ceil(e / cell)) + 2) for e in (1.0, 0.3, 1.0))
        desc = capi.hash_desc(case["mode"], (0.5, 0.0, 0.5), dims, (cell,) * 3, case["table_bits"])
        ncells = dims[0] * dims[1] * dims[2] if case["mode"] == 0 else 1 << case["table_bits"]
        dev = torch.device("cuda:0")
        out = [torch.empty(len(tris), dtype=torch.int32, device=dev) for _ in range(3)]
        out += [torch.empty(ncells, dtype=torch.int32, device=dev) for _ in range(2)]
        return dict(kind=kind, desc=desc, pos=torch.from_numpy(pos).to(dev), tris=torch.from_numpy(tris).to(dev), out=out)
    # train: strain features and the corrections they call for, as the collector records them
    X, Y = _samples(case, rng)
    ctx = capi.Context(0)
    ctx.ws_init(seed % 1000)
    ctx.ws_set_samples(X, Y)
    ctx.ws_train(0, case["batch"], 1e-3, 0)  # standardises the samples
    return dict(kind=kind, ctx=ctx, seed=seed, batch=case["batch"])


def _samples(case, rng):
    n = case["samples"]
    X = np.zeros((n, 22), np.float32)
    X[:, :3] = 0.1 * rng.standard_normal((n, 3))
    X[:, 3:21] = 0.02 * rng.standard_normal((n, 18))
    X[:, 21] = rng.random(n) < 0.01
    mix = rng.standard_normal((18, 3)) / 6.0
    Y = X[:, 3:21] @ mix + 0.05 * X[:, :3] ** 2 + 0.002 * rng.standard_normal((n, 3))
    return X, Y.astype(np.float32)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "step":
        ctx = state["ctx"]
        ctx.snapshot(True)
        ctx.step(SUBSTEPS)
        return ctx.state_save()
    if kind == "contact":
        ctx = state["ctx"]
        ctx.snapshot(True)
        ctx.step(SUBSTEPS)
        return ctx.state_save(), ctx.last_contacts()
    if kind == "detect":
        ctx = state["ctx"]
        contacts = ctx.ccd_detect(state["desc"], state["x"], state["p"], state["tris"], state["th"], state["swept"])
        m = len(contacts[0])
        for mine, new in zip(state["got"], contacts):
            mine[:m] = new
            mine[m:state["count"]] = 0
        state["count"] = m
        return m, state["got"], ctx.ccd_resolve(state["p"], state["w"], state["th"], 2)
    if kind == "hash":
        pos, tris = state["pos"], state["tris"]
        capi.check(capi.load().pbd_sh_build_noalloc(
            0, C.c_void_p(torch.cuda.current_stream().cuda_stream), C.byref(state["desc"]), C.c_void_p(pos.data_ptr()),
            len(pos), C.c_void_p(tris.data_ptr()), len(tris), *[C.c_void_p(t.data_ptr()) for t in state["out"]]))
        return state["out"]
    ctx = state["ctx"]
    ctx.ws_init(state["seed"] % 1000)
    loss = ctx.ws_train(1, state["batch"], 1e-3, state["seed"])
    return ctx.ws_params(), loss


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "detect":
        nv, nt = case["n"] ** 2, 2 * (case["n"] - 1) ** 2
        # positions, predicted positions and triangles in, resolved positions out; a cubic per triangle vertex
        return dict(bytes=float(nv * 36 + nt * 12), flops=float(300 * 3 * nt))
    if kind == "hash":
        nt = 2 * (case["n"] - 1) ** 2
        cells = 1 << case["table_bits"] if case["mode"] else nt // 2
        return dict(bytes=float(case["n"] ** 2 * 12 + nt * 24 + cells * 8), flops=float(20 * nt))
    if kind == "train":
        n = case["samples"] // case["batch"] * case["batch"] or case["samples"]
        return dict(bytes=float(n * 100 + 2 * 4 * 5827), flops=float(3 * 11392 * n))
    if kind in ("drape", "fold"):
        n = case["n"]
        ne, nb = 3 * n * n, 3 * n * n if kind == "drape" else 0
        detections = SUBSTEPS * (case["iterations"] // 10 + 1)
        nbytes = 48 * n * n + 12 * ne + 20 * nb + detections * (24 * n * n + 24 * n * n)
        cubics = detections * 6 * n * n * (9 if case["edge_edge"] else 1)
        return dict(bytes=float(nbytes), flops=float(SUBSTEPS * case["iterations"] * (28 * ne + 180 * nb) + 300 * cubics))
    nv = ne = nb = 0
    if kind == "batch":
        nv = int(case["count"] * 25800)  # mean of side^2 x aspect
        ne = 3 * nv
    else:
        rx, ry = (32, 32) if kind == "scenes" else (case["rx"], case["ry"])
        c = case["count"] if kind == "scenes" else 1
        nv, ne = c * rx * ry, c * ((ry - 1) * (3 * rx - 2) + rx - 1)
        nb = ne - 2 * (rx + ry) if case.get("bend") else 0
    # a kept cloth of a warm-started batch runs one sweep and the network
    sweeps = 1 if case.get("warm") else case["iterations"]
    flops = SUBSTEPS * (sweeps * (28 * ne + 180 * nb) + (11392 * nv if case.get("warm") else 0))
    return dict(bytes=float(48 * nv + 12 * ne + 20 * nb), flops=float(flops))


# ---------------------------------------------------------------------------
# the same outputs from plain numpy and torch in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind in ("drape", "fold", "detect", "hash") or case.get("warm"):
        # which contacts are found, which cell a centroid falls in and which
        # predictions are kept are decisions of 32-bit arithmetic at their
        # thresholds: their lists have no 64-bit value
        return None
    return _exact_frame(case, seed)


def _jittered_grid(s):
    """Grid positions with seeded jitter in 32 bits: the input of the cloth, splitmix64 per coordinate."""
    f = np.float32
    j, i = np.arange(s["rx"]), np.arange(s["ry"])
    pos = np.zeros((s["ry"], s["rx"], 3), np.float32)
    pos[:, :, 0] = j.astype(f)[None, :] * (f(s["sx"]) / f(s["rx"] - 1))
    pos[:, :, 2] = i.astype(f)[:, None] * (f(s["sy"]) / f(s["ry"] - 1))
    pos = pos.reshape(-1)
    with np.errstate(over="ignore"):
        z = np.uint64(s["seed"]) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, len(pos) + 1, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    u = f(2) * ((z >> np.uint64(40)).astype(f) * f(1.0 / 16777216.0)) - f(1)
    return (pos + f(s["jitter"]) * u).reshape(-1, 3)


def _grid_prims(rx, ry, bend):
    """Distance pairs and bending quads of a grid cloth, in their constraint order."""
    i = np.arange(rx * (ry - 1))
    col = i % rx
    right, down, diag = np.stack([i, i + 1], 1), np.stack([i, i + rx], 1), np.stack([i, i + rx - 1], 1)
    rows = np.stack([right, down, diag], 1)
    keep = np.stack([col < rx - 1, np.ones_like(col, bool), col > 0], 1)
    last = np.arange(rx * (ry - 1), rx * ry - 1)
    pairs = np.concatenate([rows[keep], np.stack([last, last + 1], 1)])
    if not bend:
        return pairs, np.zeros((0, 4), np.int64)
    t = _grid_tris(rx, ry).astype(np.int64)
    e = np.stack([t, np.roll(t, -1, 1), np.roll(t, -2, 1)], 2).reshape(-1, 3)  # (a, b, opposite) per triangle edge
    key = np.minimum(e[:, 0], e[:, 1]) * (rx * ry) + np.maximum(e[:, 0], e[:, 1])
    order = np.argsort(key, kind="stable")
    second = np.flatnonzero(key[order][1:] == key[order][:-1]) + 1
    first, second = order[second - 1], order[second]
    by = np.argsort(second, kind="stable")
    first, second = first[by], second[by]
    return pairs, np.stack([e[first, 0], e[first, 1], e[first, 2], e[second, 2]], 1)


def _colours(verts, npts, nv, dev):
    """Colours of the prims by rounds of speculative first-fit: every uncoloured prim proposes the first colour
    none of its neighbours holds and keeps it unless a neighbour of more points, or as many and a lower id,
    proposes the same.  verts: 4 vertices per prim, nv where there is none."""
    n = len(verts)
    flat = verts.reshape(-1)
    prim = torch.arange(n, device=dev).repeat_interleave(4)
    real = flat < nv
    flat, prim = flat[real], prim[real]
    order = torch.argsort(flat, stable=True)
    flat, prim = flat[order], prim[order]
    start = torch.searchsorted(flat, torch.arange(nv + 1, device=dev))
    slot = torch.arange(len(flat), device=dev) - start[flat]
    table = torch.full((nv + 1, int(slot.max()) + 1), n, dtype=torch.long, device=dev)
    table[flat, slot] = prim
    width = 4 if bool((npts == 4).any()) else 2
    colour = torch.full((n + 1,), -1, dtype=torch.long, device=dev)
    proposed = torch.full((n + 1,), -1, dtype=torch.long, device=dev)
    points = torch.cat([npts, npts.new_zeros(1)])
    act = torch.arange(n, device=dev)
    while len(act):
        nb = table[verts[act][:, :width]].reshape(len(act), -1)
        mask = torch.zeros(len(act), dtype=torch.long, device=dev)
        for k in range(nb.shape[1]):
            c = colour[nb[:, k]]
            mask |= torch.where(c >= 0, torch.ones_like(c) << c.clamp(min=0), torch.zeros_like(c))
        prop = torch.log2((~mask & (mask + 1)).double()).round().long()
        proposed[act] = prop
        proposed[n] = -1
        other = proposed[nb] == prop[:, None]
        other &= colour[nb] < 0
        mine = points[act][:, None]
        beats = (points[nb] > mine) | ((points[nb] == mine) & (nb < act[:, None]))
        lost = (other & beats).any(1)
        colour[act[~lost]] = prop[~lost]
        act = act[lost]
    return colour[:n]


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _dot(a, b):
    return (a * b).sum(1, keepdim=True)


def _hinge(q):
    e0, e1, o0, o1 = q
    E, n1, n2 = e1 - e0, _cross(o0 - e0, o0 - e1), _cross(o1 - e1, o1 - e0)
    el = _dot(E, E).sqrt()
    angle = torch.atan2(_dot(_cross(n2, n1), E) / el, _dot(n1, n2))
    return E, n1, n2, el, angle


def _exact_frame(case, seed):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    specs = _specs(case, seed)
    bend = case.get("bend", False)
    pos, pairs, quads, w, which, base = [], [], [], [], [], 0
    for k, s in enumerate(specs):
        g = _jittered_grid(s)
        a, b = _grid_prims(s["rx"], s["ry"], bend)
        wk = np.ones(len(g))
        wk[s["pins"]] = 0.0
        pos.append(g), pairs.append(a + base), quads.append(b + base), w.append(wk), which.append(np.full(len(g), k))
        base += len(g)
    to = lambda a: torch.from_numpy(np.concatenate(a)).to(dev)  # noqa: E731
    x, pairs, quads, w, which = to(pos).double(), to(pairs), to(quads), to(w)[:, None], to(which)
    v = torch.from_numpy(_velocity(seed, base)).to(dev).double()
    per = lambda f: torch.tensor([f(s) for s in specs], dtype=torch.float64, device=dev)[which]  # noqa: E731
    sphere = per(lambda s: 1.0 if s["sphere"] else 0.0)[:, None] > 0
    centre = per(lambda s: list(s["sphere"][0]) if s["sphere"] else [0.0] * 3)
    radius = per(lambda s: s["sphere"][1] if s["sphere"] else 1.0)[:, None]
    wind = per(lambda s: list(s["wind"]) if s["wind"] else [0.0] * 3)
    drag = per(lambda s: 1.0 if s["wind"] else 0.0)[:, None]
    ne, nb = len(pairs), len(quads)
    verts = torch.full((ne + nb, 4), base, dtype=torch.long, device=dev)
    verts[:ne, :2], verts[ne:] = pairs, quads
    npts = torch.full((ne + nb,), 2, dtype=torch.long, device=dev)
    npts[ne:] = 4
    colour = _colours(verts, npts, base, dev)
    length = (x[pairs[:, 0]] - x[pairs[:, 1]]).norm(dim=1, keepdim=True)
    rest = _hinge([x[quads[:, k]] for k in range(4)])[4] if nb else None
    phases = []
    for c in range(int(colour.max()) + 1):
        d, q = torch.nonzero(colour[:ne] == c)[:, 0], torch.nonzero(colour[ne:] == c)[:, 0]
        a, b = pairs[d, 0], pairs[d, 1]
        share = w[a] + w[b]
        share = torch.where(share > 0, share, torch.ones_like(share))
        phases.append((a, b, length[d], w[a] / share, w[b] / share, quads[q], rest[q] if nb else None))
    dt, sweeps = float(np.float32(DT)), case["iterations"]
    kb = 1.0 - (1.0 - float(np.float32(0.1))) ** (1.0 / sweeps)
    gravity = torch.tensor([0.0, float(np.float32(-9.8)), 0.0], dtype=torch.float64, device=dev)
    for _ in range(SUBSTEPS):
        v = v + gravity * dt * w
        v = v + (wind - v) * (drag * dt) * w
        p = x + v * dt
        for _ in range(sweeps):
            for a, b, L, wa, wb, hinge, r in phases:
                e = p[a] - p[b]
                dist = e.norm(dim=1, keepdim=True)
                step = (dist - L) * e / dist
                p[a] -= wa * step
                p[b] += wb * step
                if len(hinge):
                    q = [p[hinge[:, k]] for k in range(4)]
                    E, n1, n2, el, angle = _hinge(q)
                    s1, s2 = _dot(n1, n1), _dot(n2, n2)
                    u = [_dot(q[2] - q[1], E) / el * n1 / s1 + _dot(q[3] - q[1], E) / el * n2 / s2,
                         -(_dot(q[2] - q[0], E) / el * n1 / s1) - _dot(q[3] - q[0], E) / el * n2 / s2,
                         el / s1 * n1, el / s2 * n2]
                    den = sum(w[hinge[:, k]] * _dot(u[k], u[k]) for k in range(4))
                    ok = (den > 1e-20) & (s1 > 1e-24) & (s2 > 1e-24) & (el > 1e-12)
                    lam = torch.where(ok, (angle - r) / den * kb, torch.zeros_like(den))
                    for k in range(4):
                        p[hinge[:, k]] -= lam * w[hinge[:, k]] * u[k]
            off = p - centre
            d = off.norm(dim=1, keepdim=True)
            touch = sphere & (w > 0) & (d - radius <= 0.001) & (d > 0)
            p = torch.where(touch, p + off / d * (radius - d), p)
        v = (p - x) / dt
        x = torch.where(w >= 0, p, x)
    return x.cpu().numpy(), v.cpu().numpy()


def _splitmix(state):
    m = (1 << 64) - 1
    state = (state + 0x9E3779B97F4A7C15) & m
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return state, z ^ (z >> 31)


def _exact_train(case, seed):
    """One epoch of Adam on the 22 -> 64 -> 64 -> 3 network in 64 bits, the batches in the shuffled order."""
    X, Y = _samples(case, np.random.default_rng([seed, 79]))
    X, Y = X.astype(np.float64), Y.astype(np.float64)
    rms = lambda a: math.sqrt(float((a ** 2).mean()))  # noqa: E731
    X[:, :3] /= rms(X[:, :3])
    X[:, 3:21] /= rms(X[:, 3:21])
    X, Y = np.clip(X, -8.0, 8.0), Y / rms(Y)
    state, shapes, prm = seed % 1000, ((64, 22, 1.0), (64, 64, 1.0), (3, 64, 0.1)), []
    for rows, cols, scale in shapes:
        a, wts = scale * math.sqrt(6.0 / (rows + cols)), []
        for _ in range(rows * cols):
            state, r = _splitmix(state)
            wts.append(a * (2.0 * (r >> 40) / 16777216.0 - 1.0))
        prm += [np.array(wts).reshape(rows, cols), np.zeros(rows)]
    prm = [torch.tensor(p, dtype=torch.float64, requires_grad=True) for p in prm]
    n, batch, state = len(X), case["batch"], seed
    perm = list(range(n))
    for i in range(n - 1, 0, -1):
        state, r = _splitmix(state)
        j = r % (i + 1)
        perm[i], perm[j] = perm[j], perm[i]
    X, Y = torch.from_numpy(X)[perm], torch.from_numpy(Y)[perm]
    opt = torch.optim.Adam(prm, lr=1e-3)
    losses, first = [], 0
    while first + batch <= n or (first == 0 and n < batch):
        x, y = X[first:first + batch], Y[first:first + batch]
        for k in range(3):
            x = x @ prm[2 * k].T + prm[2 * k + 1]
            if k < 2:
                x = torch.nn.functional.gelu(x, approximate="tanh")
        loss = 0.5 * ((x - y) ** 2).sum() / len(y)
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(loss.item())
        first += batch
    return np.concatenate([p.detach().numpy().reshape(-1) for p in prm]), sum(losses) / len(losses)

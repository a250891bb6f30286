"""The calls a user of this framework makes, as measurable cases.

Each case is one pass through the public entry points: a substep (in place or
sorted, APIC or cell transfers, with the SVD or the learned closure's zero
start), a frame of graph-replayed substeps, a batch of scenes, the stage-wise
operators, a product of the implicit system, and a SparseGrid rebuilt and
sampled. Particles are generated on the device from a seed: jittered boxes or
spheres of cells as in zpc_amd/scenes.py, moving (a smooth velocity with its
gradient in C) and strained, the state a running simulation is in rather than
the one it starts from. `exact` restates each pass in 64-bit torch.
"""
import ctypes
import math
import random

import numpy as np
import torch

from zpc_amd import rocm
from zpc_amd import scenes as S

ELASTIC, SAND = S.FIXED_COROTATED, S.DRUCKER_PRAGER
GRAVITY = (0.0, -9.8, 0.0)


def listed():
    return [
        # a toy or unit-test scene: launch latency is everything
        dict(name="cube_4k", kind="substep", shape="box", a=8, b=8, c=8, cells=64, ppc=8, material="elastic",
             order="cells", driver="inplace", scheme="apic", closure=False, strain=0.02),
        # one rendered frame of the 64K-particle elastic cube: 20 substeps replayed from the captured graph
        dict(name="frame_64k", kind="frame", shape="box", a=20, b=20, c=20, cells=128, ppc=8, material="elastic",
             order="cells", steps=20, strain=0.02),
        # a small sand body of ragged size, one sorted substep (adaptive time steps take them one at a time)
        dict(name="sand_72k", kind="substep", shape="box", a=21, b=33, c=13, cells=128, ppc=8, material="sand",
             order="blocks", driver="sorted", scheme="apic", closure=False, strain=0.005),
        # the two colliding elastic spheres at dx = 1/256
        dict(name="spheres_3m8", kind="substep", shape="spheres", a=38, b=38, c=38, cells=256, ppc=8,
             material="elastic", order="blocks", driver="sorted", scheme="apic", closure=False, strain=0.02),
        # the 16,777,216-particle sand column at dx = 1/512
        dict(name="sand_16m", kind="substep", shape="box", a=128, b=256, c=64, cells=512, ppc=8, material="sand",
             order="blocks", driver="sorted", scheme="apic", closure=False, strain=0.005),
        # 64 independent scenes of 10K to 500K particles advanced by one launch per stage
        dict(name="batch_64", kind="batch", scenes=64, lo=10000, hi=500000, ppc=8, strain=0.01),
        # zpc's operators called one by one, as code written against zpc does, on particles in file order (shuffled)
        dict(name="operators_1m", kind="operators", shape="box", a=53, b=67, c=37, cells=256, ppc=8, material="sand",
             order="shuffled", strain=0.005),
        # the particle -> cell -> grid transfers
        dict(name="cell_2m", kind="substep", shape="box", a=64, b=96, c=43, cells=256, ppc=8, material="sand",
             order="cells", driver="sorted", scheme="cell", closure=False, strain=0.005),
        # one product of the implicit system (the inner step of its conjugate gradient)
        dict(name="implicit_1m", kind="implicit", shape="box", a=50, b=50, c=51, cells=256, ppc=8,
             material="elastic", order="blocks", strain=0.02),
        # a sorted substep whose stress is the learned closure's zero start, at the small strains it certifies
        dict(name="closure_4m", kind="substep", shape="box", a=80, b=101, c=65, cells=256, ppc=8, material="sand",
             order="blocks", driver="sorted", scheme="apic", closure=True, strain=0.002),
        # a level set rebuilt around the particles every frame and sampled at them
        dict(name="sparse_grid_4m", kind="sparse_grid", shape="box", a=80, b=101, c=65, cells=256, ppc=8,
             order="cells"),
    ]


def _box(rng, cells, most):
    """Odd and even box sides of at most `most` cells in all, inside the walls."""
    n = math.exp(rng.uniform(math.log(64), math.log(most)))
    side = n ** (1 / 3)
    top = cells - 12
    a = max(2, min(top, round(side * math.exp(rng.uniform(-0.5, 0.5)))))
    b = max(2, min(top, round(side * math.exp(rng.uniform(-0.5, 0.5)))))
    c = max(2, min(top, round(n / (a * b))))
    while a * b * c > most:
        a, b, c = max(2, a - 1), max(2, b - 1), max(2, c - 1)
    return a, b, c


def draw(rng):
    kind = rng.choice(["substep"] * 6 + ["frame", "frame", "batch", "operators", "implicit", "sparse_grid"])
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 64), lo=rng.randint(5000, 20000), hi=rng.randint(40000, 400000),
                    ppc=rng.randint(6, 8), strain=rng.uniform(0.005, 0.02))
    most = {"substep": 2000000, "frame": 40000, "operators": 250000, "implicit": 250000, "sparse_grid": 500000}[kind]
    cells = rng.choice([64, 128, 256, 512])
    ppc = rng.randint(4, 10)
    a, b, c = _box(rng, cells, min(most, 16000000 // ppc))
    case = dict(kind=kind, shape="box", a=a, b=b, c=c, cells=cells, ppc=ppc,
                order=rng.choice(["cells", "blocks", "shuffled"]))
    if kind == "sparse_grid":
        return case
    sand = rng.random() < 0.5
    case["material"] = "sand" if sand else "elastic"
    case["strain"] = math.exp(rng.uniform(math.log(0.002), math.log(0.05)))
    if kind == "frame":
        case.update(steps=rng.choice([2, 4, 8, 10]), material="elastic", strain=min(case["strain"], 0.02))
    if kind == "substep":
        case.update(driver=rng.choice(["inplace", "sorted", "sorted"]), scheme=rng.choice(["apic", "apic", "cell"]),
                    closure=sand and case["strain"] < 0.004 and rng.random() < 0.5)
    return case


# ---------------------------------------------------------------- particles


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _cells(g, lo, dims, dx, ppc):
    """Cell-major jittered positions, ppc per cell."""
    n = dims[0] * dims[1] * dims[2] * ppc
    cell = torch.arange(n, device="cuda") // ppc
    ijk = torch.stack([cell // (dims[1] * dims[2]), cell // dims[2] % dims[1], cell % dims[2]], 1)
    ijk += torch.tensor(lo, device="cuda")
    # 24-bit jitter short of 1, so that a particle stays in its cell
    return (ijk + torch.rand((n, 3), generator=g, device="cuda").clamp(max=0.999)).to(torch.float32) * dx


def _ball(dims, center, radius, ppc):
    """Which of the particles of _cells lie in cells whose centre is in a ball."""
    i = [torch.arange(d, device="cuda") + 0.5 - c for d, c in zip(dims, center)]
    near = i[0][:, None, None] ** 2 + i[1][:, None] ** 2 + i[2] ** 2 <= radius * radius
    return near.reshape(-1).repeat_interleave(ppc)


def _material(name, dx, ppc):
    if name == "sand":
        return S.Material.drucker_prager(3.5e5, 0.3, 1e3, 30.0, volume=dx ** 3 / ppc)
    return S.Material(kind=ELASTIC, E=1e4, nu=0.3, rho=1e3, volume=dx ** 3 / ppc)


def _dt(name, dx):
    return 5e-5 if name == "sand" and dx < 1 / 200 else 1e-4


def _keys(x, dx):
    """Block keys of float32 positions, rounded as the framework does."""
    return (torch.floor(x * float(np.float32(1) / np.float32(dx)) + 0.5).to(torch.int64) - 2) >> 2


def _pack(k):
    return ((k[..., 0] + 4096) << 40) | ((k[..., 1] + 4096) << 20) | (k[..., 2] + 4096)


def _unpack(p):
    return torch.stack([(p >> 40) - 4096, ((p >> 20) & 0xFFFFF) - 4096, (p & 0xFFFFF) - 4096], -1)


def _positions(case, g):
    cells, ppc = case["cells"], case["ppc"]
    dx = 1.0 / cells
    if case["shape"] == "spheres":
        out = []
        for cx in (0.3, 0.7):
            lo = [math.floor((p - 0.15) / dx) for p in (cx, 0.5, 0.5)]
            dims = [2 * case[k] + 2 for k in ("a", "b", "c")]
            x = _cells(g, lo, dims, dx, ppc)
            out.append(x[_ball(dims, [p / dx - q for p, q in zip((cx, 0.5, 0.5), lo)], 0.15 / dx, ppc)])
        x = torch.cat(out)
    else:
        dims = [case["a"], case["b"], case["c"]]
        lo = [(cells - dims[0]) // 2, 4, (cells - dims[2]) // 2]
        x = _cells(g, lo, dims, dx, ppc)
    if case["order"] == "blocks":  # as a sorted substep leaves them
        x = x[torch.argsort(_pack(_keys(x, dx)), stable=True)]
    elif case["order"] == "shuffled":
        x = x[torch.randperm(x.shape[0], generator=g, device="cuda")]
    return x.contiguous()


def _state(x, mat, strain, g, speed=0.5):
    """A moving, strained state at the positions x: smooth velocity, its
    gradient in C, smooth and random parts in F, some volume change in logJp."""
    n = x.shape[0]
    phase = torch.rand((3, 3), generator=g, device="cuda") * 6.28
    k = 6.0
    v, C, F = torch.zeros_like(x), torch.zeros((n, 9), device="cuda"), torch.zeros((n, 9), device="cuda")
    for d in range(3):
        for e in range(3):
            arg = k * x[:, e] + phase[d, e]
            v[:, d] += speed / 3 * torch.sin(arg)
            C[:, d + 3 * e] = speed / 3 * k * torch.cos(arg)
            F[:, d + 3 * e] = 0.5 * strain * torch.cos(2 * arg)
    F += strain * (torch.rand((n, 9), generator=g, device="cuda") - 0.5)
    F[:, ::4] += 1.0
    m = torch.full((n,), float(np.float32(mat.rho * mat.volume)), device="cuda")
    lj = strain * (torch.rand((n,), generator=g, device="cuda") - 0.5) if mat.kind == SAND else None
    return dict(x=x, v=v, C=C, F=F, m=m, logJp=lj)


def _make(case, seed):
    """(initial particle arrays, material, dx, dt) of a one-scene case."""
    g = _generator(seed)
    dx = 1.0 / case["cells"]
    mat = _material(case["material"], dx, case["ppc"])
    x = _positions(case, g)
    p = _state(x, mat, case["strain"], g)
    if case["shape"] == "spheres":
        p["v"][:, 0] += torch.where(x[:, 0] < 0.5, 2.0, -2.0)
    if case.get("scheme") == "cell":
        # the cell transfers keep B = C D in C, D the kernel's second moment per axis
        xr = x - torch.floor(x * case["cells"] + 0.5) * dx
        p["C"] *= (0.5 * (dx * dx) - xr * xr).repeat_interleave(3, dim=1)
    return p, mat, dx, _dt(case["material"], dx)


def _blocks(x, dx):
    """Packed block keys in the framework's numbering (order of first
    occurrence), the particles' blocks, and the keys the enlargement adds."""
    def numbered(p):
        u, inv = torch.unique(p, return_inverse=True)
        first = torch.full((u.shape[0],), p.shape[0], dtype=torch.int64, device=p.device)
        first.scatter_reduce_(0, inv, torch.arange(p.shape[0], device=p.device), "amin")
        order = torch.argsort(first)
        rank = torch.empty_like(order)
        rank[order] = torch.arange(order.shape[0], device=p.device)
        return u[order], rank[inv]

    keys, of = numbered(_pack(_keys(x, dx)))
    offs = torch.tensor([[i, j, k] for i in (0, 1) for j in (0, 1) for k in (0, 1)], device=x.device)
    more = _pack((_unpack(keys)[:, None, :] + offs).reshape(-1, 3))
    return numbered(torch.cat([keys, more]))[0], of


def _table_size(x, dx):
    return S.evaluate_table_size(2 * int(_blocks(x, dx)[0].shape[0]))


class _Parts:
    """Device arrays a program already holds, described for the C ABI."""

    def __init__(self, arrays, ids=False):
        n = arrays["x"].shape[0]
        self.n, self.t = n, dict(arrays)
        self.t["id"] = torch.arange(n, dtype=torch.int32, device="cuda") if ids else arrays.get("id")
        d = rocm.ParticlesDesc()
        d.hdr = rocm.Header(ctypes.sizeof(rocm.ParticlesDesc), rocm.ABI_MAJOR, rocm.ABI_MINOR)
        d.n = n
        for k in ("x", "v", "C", "F", "m", "logJp", "id"):
            t = self.t.get(k)
            setattr(d, k, None if t is None else t.data_ptr())
        self.desc = d

    def like(self):
        return _Parts({k: None if t is None else torch.zeros_like(t) for k, t in self.t.items()})

    def out(self):
        return {k: self.t[k] for k in ("x", "v", "C", "F", "logJp", "id") if self.t.get(k) is not None}


class _Scene:
    """Policy, table, grid and buckets for one set of particles."""

    def __init__(self, parts, mat, dx, dt, colliders):
        self.parts, self.dt = parts, dt
        T = _table_size(parts.t["x"], dx)
        self.pol = rocm.Policy()
        self.table = rocm.DeviceTable(T)
        self.grid = rocm.DeviceGrid(dx, max(T // 16, 64))
        self.buckets = rocm.DeviceBuckets(self.grid.cap, parts.n)
        self.model = rocm.model_desc(mat)
        self.cols = rocm.colliders_array(colliders)
        self.ncols = len(colliders)
        self.extf = (ctypes.c_float * 3)(*GRAVITY)
        self.pol.reserve(parts.n, T)

    def refs(self):
        return (ctypes.byref(self.table.desc), ctypes.byref(self.buckets.desc), ctypes.byref(self.grid.desc))

    def substep(self, out=None):
        L, r = self.pol.L, ctypes.byref
        tail = self.refs() + (self.dt, r(self.extf), self.cols, self.ncols)
        if out is None:
            rocm.check(L.zsmpm_substep__rocm(self.pol.h, r(self.model), r(self.parts.desc), *tail), "substep")
        else:
            rocm.check(L.zsmpm_substep_sorted__rocm(self.pol.h, r(self.model), r(self.parts.desc), r(out.desc), *tail),
                       "substep_sorted")

    def operators(self):
        """One substep through zpc's operators, one entry point each."""
        L, r, h = self.pol.L, ctypes.byref, self.pol.h
        t, b, gr = self.refs()
        p, m, x, n, dx = r(self.parts.desc), r(self.model), self.parts.t["x"].data_ptr(), self.parts.n, self.grid.dx
        lo, hi = (ctypes.c_int32 * 3)(0, 0, 0), (ctypes.c_int32 * 3)(2, 2, 2)
        rocm.check(L.zsmpm_table_clear__rocm(h, t), "table_clear")
        rocm.check(L.zsmpm_table_activate__rocm(h, t, x, n, dx, 4, -2, 0.5), "activate")
        rocm.check(L.zsmpm_table_enlarge__rocm(h, t, r(lo), r(hi)), "enlarge")
        rocm.check(L.zsmpm_bucket_sort__rocm(h, t, x, n, dx, 4, -2, 0.5, b), "bucket_sort")
        rocm.check(L.zsmpm_grid_clear__rocm(h, gr, t), "grid_clear")
        rocm.check(L.zsmpm_p2g__rocm(h, m, p, t, b, gr, self.dt), "p2g")
        rocm.check(L.zsmpm_grid_update__rocm(h, gr, t, self.dt, r(self.extf), self.cols, self.ncols, 1, None),
                   "grid_update")
        rocm.check(L.zsmpm_g2p__rocm(h, p, t, b, gr, self.dt), "g2p")


# ---------------------------------------------------------------- batches


def _batch(case, seed):
    """Per scene: arrays, material name, material, dx. Boxes and spheres, half
    of them sand, two grid spacings, sizes log-uniform."""
    g = _generator(seed)
    r = random.Random(case["scenes"] * 7919 + case["lo"])  # sizes belong to the case, values to the seed
    out = []
    for _ in range(case["scenes"]):
        n = math.exp(r.uniform(math.log(case["lo"]), math.log(max(case["lo"] + 1, case["hi"])))) / case["ppc"]
        ball, name, cells = r.random() < 0.5, r.choice(["sand", "elastic"]), r.choice([128, 256])
        dx = 1.0 / cells
        mat = _material(name, dx, case["ppc"])
        if ball:
            rad = (3 * n / (4 * math.pi)) ** (1 / 3)
            side = int(math.ceil(2 * rad)) + 1
        else:
            side = max(2, round(n ** (1 / 3)))
        lo = cells // 2 - side // 2
        x = _cells(g, [lo] * 3, [side] * 3, dx, case["ppc"])
        if ball:
            x = x[_ball([side] * 3, [side / 2] * 3, rad, case["ppc"])].contiguous()
        out.append((_state(x, mat, case["strain"], g), name, mat, dx))
    return out


class _BatchState:
    def __init__(self, case, seed):
        made = _batch(case, seed)
        cat = {k: torch.cat([s[0][k] for s in made]).contiguous() for k in ("x", "v", "C", "F", "m")}
        cat["logJp"] = torch.cat([s[0]["logJp"] if s[0]["logJp"] is not None else torch.zeros_like(s[0]["m"])
                                  for s in made])
        self.parts = _Parts(cat, ids=True)
        self.next = self.parts.like()
        est = sum(_table_size(s[0]["x"], s[3]) // 16 for s in made)
        T = 16 * S.next_2pow(est)
        self.pol = rocm.Policy()
        self.table = rocm.DeviceTable(T)
        self.grid = rocm.DeviceGrid(min(s[3] for s in made), max(T // 16, 64))
        self.buckets = rocm.DeviceBuckets(self.grid.cap, self.parts.n)
        self.scenes = (rocm.BatchSceneDesc * len(made))()
        first = 0
        for d, (p, name, mat, dx) in zip(self.scenes, made):
            d.hdr = rocm.Header(ctypes.sizeof(rocm.BatchSceneDesc), rocm.ABI_MAJOR, rocm.ABI_MINOR)
            d.first, d.count, d.model = first, p["x"].shape[0], rocm.model_desc(mat)
            d.dx, d.dt, d.extf = dx, _dt(name, dx), (ctypes.c_float * 3)(*GRAVITY)
            cols = S.box_walls(dx)
            d.ncolliders, d.colliders = len(cols), (rocm.PlaneCollider * rocm.MAX_COLLIDERS)(
                *rocm.colliders_array(cols))
            first += d.count
        self.pol.reserve(self.parts.n, T)

    def substep(self):
        r, in_b = ctypes.byref, ctypes.c_int32(0)
        rocm.check(self.pol.L.zsmpm_substeps_batched__rocm(
            self.pol.h, self.scenes, len(self.scenes), r(self.parts.desc), r(self.next.desc), r(self.table.desc),
            r(self.buckets.desc), r(self.grid.desc), 1, 0, r(in_b)), "substeps_batched")


# ---------------------------------------------------------------- the passes


def _host(t):
    return None if t is None else t.cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return kind, case, _BatchState(case, seed)
    if kind == "sparse_grid":
        g = _generator(seed)
        x = _positions(case, g)
        dx = 1.0 / case["cells"]
        i2w = np.diag([dx, dx, dx, 1.0])
        grid = rocm.DeviceSparseGrid(_spg_capacity(case), 1, i2w, background=4 * dx)
        grid.data.copy_(_spg_values(grid.data.shape, g))
        return kind, case, (grid, x)
    p, mat, dx, dt = _make(case, seed)
    if kind == "frame" or (kind == "substep" and case["driver"] == "inplace" and p["x"].shape[0] < 100000):
        # a small scene goes through the Python driver
        sc = S.Scene("case", dx, dt, mat, *(_host(p[k]) for k in ("x", "v", "C", "F", "m", "logJp")),
                     gravity=GRAVITY, colliders=S.box_walls(dx), table_size=_table_size(p["x"], dx))
        sim = rocm.Simulator(sc, reorder=kind == "frame")
        if kind == "frame":
            start = {k: getattr(sim.parts, k).clone() for k in ("x", "v", "C", "F", "m", "logJp", "id")
                     if getattr(sim.parts, k) is not None}
            return kind, case, (sim, start)
        sim.pol.set_transfer_scheme(rocm.TRANSFER_CELL if case["scheme"] == "cell" else rocm.TRANSFER_APIC)
        if case["closure"]:
            sim.pol.set_closure(None)
        return "simulator", case, sim
    parts = _Parts(p, ids=kind == "substep" and case["driver"] == "sorted")
    sc = _Scene(parts, mat, dx, dt, S.box_walls(dx))
    if kind == "substep":
        sc.pol.set_transfer_scheme(rocm.TRANSFER_CELL if case["scheme"] == "cell" else rocm.TRANSFER_APIC)
        if case["closure"]:
            sc.pol.set_closure(None)
        return kind, case, (sc, parts.like() if case["driver"] == "sorted" else None)
    if kind == "implicit":
        # the table, the node masses and a velocity field: what the time step has before its solve
        L, r, h = sc.pol.L, ctypes.byref, sc.pol.h
        t, b, gr = sc.refs()
        lo, hi = (ctypes.c_int32 * 3)(0, 0, 0), (ctypes.c_int32 * 3)(2, 2, 2)
        rocm.check(L.zsmpm_table_clear__rocm(h, t), "table_clear")
        rocm.check(L.zsmpm_table_activate__rocm(h, t, p["x"].data_ptr(), parts.n, dx, 4, -2, 0.5), "activate")
        rocm.check(L.zsmpm_table_enlarge__rocm(h, t, r(lo), r(hi)), "enlarge")
        rocm.check(L.zsmpm_grid_clear__rocm(h, gr, t), "grid_clear")
        rocm.check(L.zsmpm_p2g__rocm(h, r(sc.model), r(parts.desc), t, None, gr, dt), "p2g")
        sc.pol.sync()
        v = _field(_blocks(p["x"], dx)[0], sc.grid.cap, dx)
        return kind, case, (sc, v, torch.zeros_like(v))
    return kind, case, sc


def run(state):
    kind, case, s = state
    if kind == "batch":
        s.substep()
        return s.next.out()
    if kind == "simulator":
        s.substep()
        return {k: getattr(s.parts, k) for k in ("x", "v", "C", "F", "logJp") if getattr(s.parts, k) is not None}
    if kind == "frame":
        # every frame starts from the state the program keeps, and is read by particle id
        sim, start = s
        for k, t in start.items():
            getattr(sim.parts, k).copy_(t)
        sim.substeps(case["steps"], graph=True)
        ids = sim.parts.id.long()
        out = {k: torch.empty_like(start[k]) for k in ("x", "v", "C", "F")}
        for k, t in out.items():
            t.index_copy_(0, ids, getattr(sim.parts, k))
        return out
    if kind == "substep":
        sc, out = s
        sc.substep(out)
        return (out or sc.parts).out()
    if kind == "operators":
        s.operators()
        return {**s.parts.out(), "indices": s.buckets.indices, "counts": s.buckets.counts, "keys": s.table.keys}
    if kind == "implicit":
        sc, v, out = s
        r = ctypes.byref
        rocm.check(sc.pol.L.zsmpm_implicit_multiply__rocm(
            sc.pol.h, r(sc.model), r(sc.parts.desc), r(sc.table.desc), r(sc.grid.desc), sc.dt, v.data_ptr(),
            out.data_ptr()), "implicit_multiply")
        return out
    grid, x = s
    grid.table.clear()
    grid.activate(x)
    return {"values": grid.sample(0, x), "count": grid.table.cnt, "keys": grid.table.keys}


def work(case):
    """Bytes: every particle attribute the pass reads and every one it leaves,
    once. Flops: per particle, two 27-node transfers and the stress."""
    if case["kind"] == "batch":
        n = 0.0
        for s in _batch_sizes(case):
            n += s
        return {"bytes": n * (108 + 108), "flops": n * 2600}
    n = _count(case)
    sand = case.get("material") == "sand"
    state = 104 if sand else 100
    if case["kind"] == "frame":
        return {"bytes": n * case["steps"] * 2.0 * state, "flops": n * case["steps"] * 2600.0}
    if case["kind"] == "implicit":
        # positions, F and masses in; the vector of the occupied nodes in and out
        return {"bytes": n * 52.0 + 24.0 * n / case["ppc"], "flops": n * 2600.0}
    if case["kind"] == "sparse_grid":
        return {"bytes": n * (12.0 + 4.0) + 4.0 * n / case["ppc"], "flops": n * 60.0}
    ids = 8 if case.get("driver") == "sorted" else 0
    return {"bytes": n * (2.0 * state + ids), "flops": n * 2600.0}


def _count(case):
    if case["shape"] == "spheres":
        return 2 * 4 / 3 * math.pi * (0.15 * case["cells"]) ** 3 * case["ppc"]
    return float(case["a"] * case["b"] * case["c"] * case["ppc"])


def _batch_sizes(case):
    r = random.Random(case["scenes"] * 7919 + case["lo"])
    for _ in range(case["scenes"]):
        n = math.exp(r.uniform(math.log(case["lo"]), math.log(max(case["lo"] + 1, case["hi"]))))
        r.random(), r.choice([0, 1]), r.choice([128, 256])
        yield n


def _spg_capacity(case):
    """Blocks of 8^3 voxels a level set around the body may take, with room."""
    nb = 1
    for k in ("a", "b", "c"):
        nb *= case[k] // 8 + 3
    return 2 * nb


def _spg_values(shape, g):
    return torch.rand(shape, generator=g, device="cuda") - 0.5


def _field(keys, cap, dx):
    """A smooth velocity at the nodes of the blocks, 3 floats per node, zero beyond them."""
    cell = torch.arange(64, device="cuda")
    node = 4 * _unpack(keys)[:, None, :] + torch.stack([cell >> 4, (cell >> 2) & 3, cell & 3], 1)
    pos = (node * dx).to(torch.float32).reshape(-1, 3)
    v = torch.zeros((cap * 64, 3), device="cuda")
    for d in range(3):
        v[:pos.shape[0], d] = 0.4 * torch.sin(6 * pos[:, d] + 5 * pos[:, (d + 1) % 3]) + 0.1
    return v.reshape(-1)


# ---------------------------------------------------------------- 64-bit restatement


def _mm(A, B):
    return (A.unsqueeze(-1) * B.unsqueeze(-3)).sum(-2)


def _eigen(b):
    """Eigenvalues and vectors (columns) of symmetric 3x3 matrices: cyclic Jacobi."""
    s = [[b[:, i, j] for j in range(3)] for i in range(3)]
    one, zero = torch.ones_like(s[0][0]), torch.zeros_like(s[0][0])
    v = [[one if i == j else zero for j in range(3)] for i in range(3)]
    for _ in range(7):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            r = 3 - p - q
            off = s[p][q]
            safe = torch.where(off == 0, one, off)
            th = (s[q][q] - s[p][p]) / (2 * safe)
            t = torch.where(th >= 0, one, -one) / (th.abs() + torch.sqrt(th * th + 1))
            t = torch.where(off == 0, zero, t)
            c = 1 / torch.sqrt(t * t + 1)
            sn = t * c
            s[p][p], s[q][q] = s[p][p] - t * off, s[q][q] + t * off
            s[p][q] = s[q][p] = zero
            rp, rq = s[r][p], s[r][q]
            s[r][p] = s[p][r] = c * rp - sn * rq
            s[r][q] = s[q][r] = sn * rp + c * rq
            for i in range(3):
                v[i][p], v[i][q] = c * v[i][p] - sn * v[i][q], sn * v[i][p] + c * v[i][q]
    return (torch.stack([s[i][i] for i in range(3)], 1),
            torch.stack([torch.stack(row, 1) for row in v], 1))


def _det(F):
    return (F[:, 0, 0] * (F[:, 1, 1] * F[:, 2, 2] - F[:, 1, 2] * F[:, 2, 1])
            - F[:, 0, 1] * (F[:, 1, 0] * F[:, 2, 2] - F[:, 1, 2] * F[:, 2, 0])
            + F[:, 0, 2] * (F[:, 1, 0] * F[:, 2, 1] - F[:, 1, 1] * F[:, 2, 0]))


def _stress64(mat, F, lj):
    """vol P F^T and the new logJp: both models act on b = F F^T's principal values."""
    f = np.float32
    E, nu, vol = float(f(mat.E)), float(f(mat.nu)), float(f(mat.volume))
    mu, lam = 0.5 * E / (1 + nu), E * nu / ((1 + nu) * (1 - 2 * nu))
    w, U = _eigen(_mm(F, F.transpose(1, 2)))
    sig = torch.sqrt(w.clamp(min=0))
    if mat.kind == ELASTIC:
        J = _det(F)
        low = torch.zeros_like(sig).scatter_(1, sig.argmin(1, keepdim=True), 1.0)
        sig = torch.where((low > 0) & (J[:, None] < 0), -sig, sig)
        tau = 2 * mu * (sig - 1) * sig + (lam * (J - 1) * J)[:, None]
    else:
        coh, beta, ys = float(f(mat.cohesion)), float(f(mat.beta)), float(f(mat.yield_surface))
        eps = torch.log(sig.clamp(min=1e-4)) - coh
        tot = eps.sum(1)
        tr = tot + lj
        dev = eps - (tr / 3)[:, None]
        norm = torch.sqrt((dev * dev).sum(1))
        dg = norm + (3 * lam + 2 * mu) / (2 * mu) * tr * ys
        back = (dg / torch.where(norm == 0, torch.ones_like(norm), norm))[:, None] * dev
        H = eps - torch.where(dg[:, None] > 0, back, torch.zeros_like(back)) + coh
        H = torch.where(tr[:, None] >= 0, torch.full_like(H, coh), H)
        lj = torch.where(tr >= 0, beta * tot + lj, torch.zeros_like(lj))
        tau = 2 * mu * H + (lam * H.sum(1))[:, None]
    return vol * _mm(U * tau[:, None, :], U.transpose(1, 2)), lj


def _weights64(x, dx, scheme):
    X = x / dx
    base = torch.floor(X - 0.5).to(torch.int64)
    l = X - base
    if scheme == "cell":
        t = l - 0.5
        w = [(1 - t) / 2, torch.full_like(t, 0.5), t / 2]
        xr = x - torch.floor(X + 0.5) * dx
        dinv = 2 / (dx * dx - 2 * xr * xr)
    else:
        w = [0.5 * (1.5 - l) ** 2, 0.75 - (l - 1) ** 2, 0.5 * (l - 0.5) ** 2]
        dinv = torch.full_like(x, 4 / (dx * dx))
    return base, l, w, dinv


class _Grid64:
    """Dense nodes over the particles' stencils."""

    def __init__(self, base):
        self.lo = base.amin(0)
        self.dims = [int(v) for v in (base.amax(0) - self.lo + 3)]
        self.size = self.dims[0] * self.dims[1] * self.dims[2]

    def at(self, node):
        r = node - self.lo
        return (r[..., 0] * self.dims[1] + r[..., 1]) * self.dims[2] + r[..., 2]

    def holds(self, node):
        r = node - self.lo
        return ((r >= 0) & (r < torch.tensor(self.dims, device=r.device))).all(-1)

    def nodes(self):
        i = torch.arange(self.size, device="cuda")
        return torch.stack([i // (self.dims[1] * self.dims[2]), i // self.dims[2] % self.dims[1],
                            i % self.dims[2]], 1) + self.lo


def _each(w, base, grid):
    at = grid.at(base)
    for a in range(3):
        for b in range(3):
            wab = w[a][:, 0] * w[b][:, 1]
            for c in range(3):
                yield wab * w[c][:, 2], (a, b, c), at + (a * grid.dims[1] + b) * grid.dims[2] + c


def _substep64(p, mat, dx, dt, scheme="apic"):
    """One substep of 64-bit arrays (x, v, C, F as 3x3, m, logJp), in place order."""
    dt = float(np.float32(dt))
    x, v, C, F, m = p["x"], p["v"], p["C"], p["F"], p["m"]
    PF, lj = _stress64(mat, F, p.get("logJp"))
    base, l, w, dinv = _weights64(x, dx, scheme)
    g = _Grid64(base)
    A = (m[:, None, None] * C * (dinv[:, None, :] if scheme == "cell" else 1.0) - dt * PF * dinv[:, None, :]) * dx
    val = torch.empty((x.shape[0], 4), dtype=torch.float64, device="cuda")
    acc = torch.zeros((g.size, 4), dtype=torch.float64, device="cuda")
    B = m[:, None] * v - (A * l[:, None, :]).sum(2)
    for W, (a, b, c), at in _each(w, base, g):
        val[:, 0] = W * m
        val[:, 1:] = W[:, None] * (B + a * A[:, :, 0] + b * A[:, :, 1] + c * A[:, :, 2])
        acc.index_add_(0, at, val)
    del val, A, B, PF
    vel = acc[:, 1:] / torch.where(acc[:, :1] == 0, torch.ones_like(acc[:, :1]), acc[:, :1])
    vel = vel + dt * torch.tensor([float(np.float32(k)) for k in GRAVITY], dtype=torch.float64, device="cuda")
    pos = g.nodes().double() * dx
    for col in S.box_walls(dx):
        o = torch.tensor(col.origin, dtype=torch.float64, device="cuda")
        nrm = torch.tensor(col.normal, dtype=torch.float64, device="cuda")
        vel[((pos - o) * nrm).sum(1) < 0] = 0
    nv, nC = torch.zeros_like(v), torch.zeros_like(C)
    for W, o, at in _each(w, base, g):
        vi = W[:, None] * vel[at]
        nv += vi
        nC += vi[:, :, None] * ((torch.tensor(o, dtype=torch.float64, device="cuda") - l) * dx)[:, None, :]
    scaled = nC * dinv[:, None, :]
    return dict(x=x + dt * nv, v=nv, C=nC if scheme == "cell" else scaled, F=F + dt * _mm(scaled, F), m=m, logJp=lj)


def _to64(p):
    q = {k: None if t is None else t.double() for k, t in p.items()}
    for k in ("C", "F"):
        q[k] = q[k].reshape(-1, 3, 3).transpose(1, 2)
    return q


def _flat(p, keys=("x", "v", "C", "F", "logJp")):
    out = {}
    for k in keys:
        if p.get(k) is not None:
            out[k] = p[k].transpose(1, 2).reshape(-1, 9) if k in ("C", "F") else p[k]
    return out


def _sorted64(p, x32, dx):
    perm = torch.argsort(_blocks(x32, dx)[1], stable=True)
    return {k: t[perm] for k, t in p.items()}


def _multiply64(case, seed):
    p, mat, dx, dt = _make(case, seed)
    dt = float(np.float32(dt))
    q = _to64(p)
    keys = _blocks(p["x"], dx)[0]
    cap = max(_table_size(p["x"], dx) // 16, 64)
    v = _field(keys, cap, dx).double().reshape(-1, 3)
    base, l, w, dinv = _weights64(q["x"], dx, "apic")
    g = _Grid64(base)
    cell = torch.arange(64, device="cuda")
    node = (4 * _unpack(keys)[:, None, :] + torch.stack([cell >> 4, (cell >> 2) & 3, cell & 3], 1)).reshape(-1, 3)
    held = g.holds(node)
    vel = torch.zeros((g.size, 3), dtype=torch.float64, device="cuda")
    vel[g.at(node)[held]] = v[:node.shape[0]][held]
    C = torch.zeros_like(q["C"])
    for W, o, at in _each(w, base, g):
        off = (torch.tensor(o, dtype=torch.float64, device="cuda") - l) * dx
        C += (W[:, None] * vel[at])[:, :, None] * (off * dinv)[:, None, :]
    PF, _ = _stress64(mat, q["F"] + dt * _mm(C, q["F"]), q.get("logJp"))
    acc = torch.zeros((g.size, 4), dtype=torch.float64, device="cuda")
    for W, o, at in _each(w, base, g):
        off = (torch.tensor(o, dtype=torch.float64, device="cuda") - l) * dx
        f = (PF * (off * dinv)[:, None, :]).sum(2) * W[:, None]
        acc.index_add_(0, at, torch.cat([(W * q["m"])[:, None], f], 1))
    out = torch.zeros_like(v)
    at = g.at(node)[held]
    full = (acc[at, 1:] * dt * dt + acc[at, :1]) * v[:node.shape[0]][held]
    out[:node.shape[0]][held] = torch.where(acc[at, :1] > 0, full, acc[at, 1:])
    return out.reshape(-1)


def _sample64(case, seed):
    g = _generator(seed)
    x = _positions(case, g)
    dx = 1.0 / case["cells"]
    vals = _spg_values((_spg_capacity(case), 1, 512), g).double()[:, 0]
    X = x.double() * float(np.float32(1.0 / dx))
    key = torch.floor(x * float(np.float32(1.0 / dx)) + 0.5).to(torch.int64)
    p = _pack(key >> 3)
    u, inv = torch.unique(p, return_inverse=True)
    first = torch.full((u.shape[0],), p.shape[0], dtype=torch.int64, device="cuda")
    first.scatter_reduce_(0, inv, torch.arange(p.shape[0], device="cuda"), "amin")
    rank = torch.empty_like(first)
    rank[torch.argsort(first)] = torch.arange(first.shape[0], device="cuda")
    lo = torch.floor(X).to(torch.int64)
    fr = X - lo
    out = torch.zeros_like(fr[:, 0])
    for a in range(2):
        for b in range(2):
            for c in range(2):
                n = lo + torch.tensor([a, b, c], device="cuda")
                q = _pack(n >> 3)
                j = torch.searchsorted(u, q).clamp(max=u.shape[0] - 1)
                k = ((n[:, 0] & 7) * 8 + (n[:, 1] & 7)) * 8 + (n[:, 2] & 7)
                val = torch.where(u[j] == q, vals[rank[j], k], torch.full_like(out, float(np.float32(4 * dx))))
                w = (fr[:, 0] if a else 1 - fr[:, 0]) * (fr[:, 1] if b else 1 - fr[:, 1])
                out += val * w * (fr[:, 2] if c else 1 - fr[:, 2])
    return {"values": out, "count": None, "keys": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "sparse_grid":
        return _sample64(case, seed)
    if kind == "implicit":
        return _multiply64(case, seed)
    if kind == "batch":
        parts = []
        for p, name, mat, dx in _batch(case, seed):
            q = _substep64(_to64(p), mat, dx, _dt(name, dx))
            if q["logJp"] is None:
                q["logJp"] = torch.zeros_like(q["m"])
            parts.append(_flat(_sorted64(q, p["x"], dx)))
        return {**{k: torch.cat([q[k] for q in parts]) for k in parts[0]}, "id": None}
    p, mat, dx, dt = _make(case, seed)
    q = _to64(p)
    if kind == "frame":
        for _ in range(case["steps"]):
            q = _substep64(q, mat, dx, dt)
        return _flat(q, ("x", "v", "C", "F"))
    q = _substep64(q, mat, dx, dt, case.get("scheme", "apic"))
    if q["logJp"] is None:
        del q["logJp"]
    if kind == "operators":
        return {**_flat(q), "indices": None, "counts": None, "keys": None}
    if case["driver"] == "sorted":
        return {**_flat(_sorted64(q, p["x"], dx)), "id": None}
    return _flat(q)

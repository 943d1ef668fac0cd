"""What a user of the shallow-water patch path has it do, as timed cases.

Each case is one pass through the public entry points on state that stays on
the GPU between passes, as it does in a simulation:

* ``grid``    `PatchPool.step` / `graph_replay` of a uniform grid of patches
              (radial dam break over hills, or the wet/dry basin), f-wave or
              augmented Riemann solver, every CFL mode
* ``uneven``  the batched step of many patches of 8^2 .. 64^2 cells
* ``amr``     `BatchedAmr.step` of a 2- or 3-level adaptive grid
* ``lts``     `BatchedAmr.lts_iterations`, local time stepping on the same
* ``calls``   one grid iteration made of single `Numerics` calls
              (`AmrGrid.step` on a `DeviceBackend`), as a Peano host makes them
* ``regrid``  the data work of a regrid: refinement flags, interpolation into
              new patches, restriction into coarsened ones
* ``serve``   `Server`: independent requests admitted, stepped together and
              retired

`exact` advances the same inputs in plain torch (64 bits) on whole batches of
tiles; it shares no code with the package.
"""
import ctypes
import math
import random

import numpy as np
import torch

from peanoclaw_amd.amr import AmrGrid, BatchedAmr, DeviceBackend
from peanoclaw_amd.pool import PatchPool, make_description, tile_stride
from peanoclaw_amd.scenarios import GridLayout, Workload
from peanoclaw_amd.serving import Server, make_request

GRAVITY = 9.81
DRY = 0.01
ZERO = 1e-7
EPS = 1e-8
CFL = 0.4
SIZES = (64, 32, 16, 8)  # patch classes of the uneven workload
SERVE_PATCH = 32         # cells per patch side of a served request
SERVE_ROUND = 64         # steps per server round
DEV = "cuda"
F64 = torch.float64


def listed():
    return [
        # the smallest configuration: 9 x 9 patches of 16^2, radial dam break
        # on a flat bottom; launches and latency decide
        {"name": "dam_9x9x16", "kind": "grid", "data": "dam", "px": 9, "py": 9, "nx": 16,
         "ny": 16, "hills": 0, "fused": 2, "solver": 1, "form": "step", "steps": 20},
        # a served-size grid stepped from a captured graph
        {"name": "dam_24x24x32_graph", "kind": "grid", "data": "dam", "px": 24, "py": 24,
         "nx": 32, "ny": 32, "hills": 5, "fused": 2, "solver": 1, "form": "graph", "steps": 20},
        # a large uniform grid (2560^2 cells)
        {"name": "dam_40x40x64", "kind": "grid", "data": "dam", "px": 40, "py": 40, "nx": 64,
         "ny": 64, "hills": 5, "fused": 2, "solver": 1, "form": "step", "steps": 10},
        # the headline workload: 50,000 patches of 8^2 .. 64^2 in one step
        {"name": "uneven_50k", "kind": "uneven", "patches": 50000, "fused": 2, "steps": 2},
        # wet/dry basin with the pool as created (exact speed pass each step)
        {"name": "basin_27x27x27", "kind": "grid", "data": "basin", "px": 27, "py": 27,
         "nx": 27, "ny": 27, "hills": 6, "fused": 0, "solver": 1, "form": "step", "steps": 10},
        # the same physics with the augmented Riemann solver
        {"name": "basin_16x16x32_augmented", "kind": "grid", "data": "basin", "px": 16,
         "py": 16, "nx": 32, "ny": 32, "hills": 6, "fused": 0, "solver": 2, "form": "step",
         "steps": 10},
        # 2-level dam break, the ten steps between two regrids
        {"name": "amr_27x27x16_2_levels", "kind": "amr", "data": "dam", "px": 27, "n": 16,
         "levels": 2, "steps": 10},
        # 3-level wet/dry basin of 2187^2 effective cells
        {"name": "amr_9x9x27_3_levels", "kind": "amr", "data": "basin", "px": 9, "n": 27,
         "levels": 3, "steps": 10},
        # local time stepping on the 2-level grid, one batch of iterations
        {"name": "lts_27x27x16_2_levels", "kind": "lts", "data": "dam", "px": 27, "n": 16,
         "levels": 2, "steps": 16},
        # a Peano host's grid iteration: every Numerics call by itself
        {"name": "calls_3x3x16_2_levels", "kind": "calls", "data": "dam", "px": 3, "n": 16,
         "levels": 2, "steps": 1},
        # a regrid of a medium adaptive grid: 24 patches refined, 24 coarsened
        {"name": "regrid_24x16", "kind": "regrid", "parents": 24, "n": 16},
        # a burst of independent requests until all have finished
        {"name": "serve_8_requests", "kind": "serve", "requests": 8, "n_min": 64, "n_max": 512,
         "end_time": 0.1},
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["grid", "grid", "grid", "uneven", "amr", "amr", "lts", "calls", "regrid",
                       "serve"])
    if kind == "grid":
        data = rng.choice(["dam", "dam", "basin"])
        solver = rng.choice([1, 1, 2])
        nx = rng.randint(8, 64)
        ny = nx if rng.random() < 0.5 else rng.randint(8, 64)
        cells = math.exp(rng.uniform(math.log(4e3), math.log(1.6e7 if solver == 1 else 1e6)))
        px = max(1, int(round(math.sqrt(cells) / nx)))
        py = max(1, int(round(math.sqrt(cells) / ny)))
        return {"kind": kind, "data": data, "px": px, "py": py, "nx": nx, "ny": ny,
                "hills": rng.randint(0, 8) if data == "dam" else 6,
                "fused": rng.choice([0, 1, 2, 2]), "solver": solver,
                "form": rng.choice(["step", "graph"]),
                "steps": 2 * rng.randint(1, 10) if cells < 2e6 else 2}
    if kind == "uneven":
        return {"kind": kind, "patches": _log_int(rng, 300, 40000), "fused": 2, "steps": 2}
    if kind in ("amr", "lts"):
        levels = rng.choice([2, 2, 3])
        n = rng.randint(8, 32)
        px = rng.randint(4, 27 if levels == 2 else 9)
        return {"kind": kind, "data": rng.choice(["dam", "basin"]), "px": px, "n": n,
                "levels": levels, "steps": rng.randint(1, 20)}
    if kind == "calls":
        return {"kind": kind, "data": "dam", "px": rng.randint(2, 4), "n": rng.randint(8, 64),
                "levels": rng.choice([1, 2]), "steps": 1}
    if kind == "regrid":
        return {"kind": kind, "parents": _log_int(rng, 1, 150), "n": rng.randint(6, 48)}
    return {"kind": kind, "requests": rng.randint(1, 8), "n_min": 64,
            "n_max": 32 * rng.randint(2, 20), "end_time": rng.choice([0.02, 0.05, 0.1])}


# ---- initial data (functions of the cell centres, numpy or torch) ----

def _rng(case, seed):
    return random.Random("%s/%d" % (case["kind"], seed))


def _dam(rng, hills, inner):
    """Radial column of depth `inner` (jittered centre) over Gaussian hills."""
    cx, cy = (0.5 + rng.uniform(-0.05, 0.05) for _ in range(2))
    bumps = [(rng.uniform(0, 1), rng.uniform(0, 1), rng.uniform(0.05, 0.15),
              rng.uniform(0.0, 0.3)) for _ in range(hills)]

    def fn(X, Y, xp=np):
        r = xp.sqrt((X - cx) ** 2 + (Y - cy) ** 2)
        b = 0.0 * r
        h = xp.where(r <= 0.25, b + inner, b + 1.0)
        for x, y, s, a in bumps:
            b = b + a * xp.exp(-((X - x) ** 2 + (Y - y) ** 2) / (s * s))
        return h, b
    return fn


def _basin(rng, hills, depth):
    """Sloping basin with bumps, still water at level 0 where b < 0, dry land
    elsewhere, and a column of depth `depth` over 10 % of the domain."""
    bumps = [(rng.uniform(0.2, 0.9), rng.uniform(0.1, 0.9), rng.uniform(0.03, 0.1),
              rng.uniform(-0.15, 0.15)) for _ in range(hills)]

    def fn(X, Y, xp=np):
        b = -1.0 + 1.5 * X
        for x, y, s, a in bumps:
            b = b + a * xp.exp(-((X - x) ** 2 + (Y - y) ** 2) / (2 * s * s))
        h = xp.where(b < 0.0, -b, 0.0 * b)
        col = (X >= 0.05) & (X <= 0.35) & (Y >= 0.3) & (Y <= 0.3 + 0.1 / 0.3)
        return xp.where(col, 0.0 * h + depth, h), b
    return fn


def _field_fn(case, seed):
    # an adaptive grid's tree belongs to the case: only the column's depth
    # comes from the seed there
    geometry = _rng(case, seed if case["kind"] == "grid" else 0)
    jitter = _rng(case, seed).uniform(-0.1, 0.1)
    if case["data"] == "basin":
        return _basin(geometry, 6, 1.5 + jitter)
    return _dam(geometry, case.get("hills", 0), 2.0 + jitter)


def _centres(pos, size, n):
    """Cell centres, ghost ring included, of tiles at pos (k, 2): X (k, n+2, 1)
    and Y (k, 1, n+2)."""
    ii = torch.arange(-1, n[0] + 1, dtype=F64, device=DEV) + 0.5
    jj = torch.arange(-1, n[1] + 1, dtype=F64, device=DEV) + 0.5
    pos = torch.as_tensor(np.asarray(pos, dtype=np.float64).reshape(-1, 2), device=DEV)
    return (pos[:, 0, None, None] + ii[None, :, None] * (size[0] / n[0]),
            pos[:, 1, None, None] + jj[None, None, :] * (size[1] / n[1]))


def _grid_tiles(case, seed):
    """(h, hu, hv, b) of every patch of a grid case, and its geometry."""
    px, py, n = case["px"], case["py"], (case["nx"], case["ny"])
    size = (1.0 / px, 1.0 / py)
    pos = [(i * size[0], j * size[1]) for i in range(px) for j in range(py)]
    X, Y = torch.broadcast_tensors(*_centres(pos, size, n))
    h, b = _field_fn(case, seed)(X, Y, torch)
    z = torch.zeros_like(h)
    return [h, z, z.clone(), b], pos, size, n


def _uneven_counts(case):
    kinds = np.random.default_rng(2).integers(0, len(SIZES), case["patches"])
    return {n: int((kinds == k).sum()) for k, n in enumerate(SIZES)}


def _uneven_tiles(case, seed):
    """Per size class its tiles, tiled column by column into a grid whose last
    column may be partly empty: noise plus bumps in h, small momenta, hills."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    rng = _rng(case, seed)
    dx = 1.0 / 64
    out = []
    for n, count in _uneven_counts(case).items():
        if not count:
            continue
        width = int(math.ceil(math.sqrt(count)))
        rows = -(-count // width)
        span = (width * n * dx, rows * n * dx)
        big = max(span)
        pos = [((k // rows) * n * dx, (k % rows) * n * dx) for k in range(count)]
        X, Y = torch.broadcast_tensors(*_centres(pos, (n * dx, n * dx), (n, n)))

        def gauss(k, s0, s1, a0, a1):
            f = torch.zeros_like(X)
            for _ in range(k):
                x, y = rng.uniform(0, span[0]), rng.uniform(0, span[1])
                s, a = big * rng.uniform(s0, s1), rng.uniform(a0, a1)
                f += a * torch.exp(-((X - x) ** 2 + (Y - y) ** 2) / (2 * s * s))
            return f

        def noise(lo, hi):
            return torch.rand(X.shape, generator=gen, dtype=F64, device=DEV) * (hi - lo) + lo
        h = torch.clamp(0.8 + 0.2 * noise(0.0, 1.0) + gauss(3, 0.05, 0.2, 0.2, 0.5), 0.5, 2.0)
        out.append(([h, noise(-0.1, 0.1), noise(-0.1, 0.1), gauss(5, 0.05, 0.15, 0.0, 0.3)],
                    pos, n, dx, width, rows))
    return out


# ---- the pool's arrays as torch tensors ----

class _Array:
    """One field array; a tensor made of it keeps the pool open."""

    def __init__(self, pool, ptr, cells):
        self.pool = pool
        self.__cuda_array_interface__ = {"shape": (cells,), "typestr": "<f8", "version": 3,
                                         "data": (ptr, False), "strides": None}


def _fields(pool, state, cells):
    """h, hu, hv (of one state) and b of the pool, flat, without a copy."""
    p = [ctypes.POINTER(ctypes.c_double)() for _ in range(4)]
    if pool.lib.pc_pool_device_fields(pool.h, state, *(ctypes.byref(q) for q in p)):
        raise RuntimeError("pc_pool_device_fields")
    return [torch.as_tensor(_Array(pool, ctypes.cast(q, ctypes.c_void_p).value, cells),
                            device=DEV) for q in p]


def _tiles(pool, first, count, n, state, ring):
    """Views (count, n, n) of h, hu, hv, b of `count` consecutive tiles, with
    or without the ghost ring."""
    stride = tile_stride(n[1])
    per = (n[0] + 2) * stride
    off = pool.offset(first)
    if ring:
        shape, start = (count, n[0] + 2, n[1] + 2), off
    else:
        shape, start = (count, n[0], n[1]), off + stride + 1
    return [f.as_strided(shape, (per, stride, 1), start)
            for f in _fields(pool, state, off + per * count)]


def _register(pool, pos, size, n, **kw):
    slots = [pool.register(make_description(p, size, n[0], ny=n[1], **kw)) for p in pos]
    per = (n[0] + 2) * tile_stride(n[1])
    if any(pool.offset(s) != pool.offset(slots[0]) + k * per for k, s in enumerate(slots)):
        raise RuntimeError("tiles are not consecutive")
    return slots


def _reserve(pool, tiles):
    pool.reserve(sum(c * ((n[0] + 2) * tile_stride(n[1]) + 16) for c, n in tiles))


def _write(pool, slots, n, state, values):
    pool.synchronize()
    for dst, src in zip(_tiles(pool, slots[0], len(slots), n, state, True), values):
        if src is not None:
            dst.copy_(src)
    torch.cuda.synchronize()


class State:
    """What a program keeps between passes.  The pool itself closes when the
    last output that views it is gone."""

    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)

    def __del__(self):
        for name in ("amr", "server"):
            if name in self.__dict__:
                self.__dict__[name].close()


# ---- prepare ----

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _stepping(pool, case, layouts, views):
    wl = Workload(pool, layouts, 0, 0, [])
    pool.scenario_set(0, 0.0, 0.0, np.inf)
    wl.build_ghost_table()
    pool.wave_propagation_solver(case.get("solver", 1))
    pool.launch_config(fused=case["fused"])
    if case.get("form") == "graph":
        pool.graph_capture()
    return State(case, pool=pool, views=views)


def _prepare_grid(case, seed):
    values, pos, size, n = _grid_tiles(case, seed)
    pool = PatchPool(0)
    _reserve(pool, [(len(pos), n)])
    slots = _register(pool, pos, size, n)
    _write(pool, slots, n, pool.current_state(0), values)
    layout = GridLayout(n[0], np.array(slots, dtype=np.int32).reshape(case["px"], case["py"]),
                        n[1])
    # an even number of steps ends in the state it began in
    views = _tiles(pool, slots[0], len(slots), n, pool.current_state(0), False)[:3]
    return _stepping(pool, case, [layout], {"h": views[0], "hu": views[1], "hv": views[2]})


def _prepare_uneven(case, seed):
    classes = _uneven_tiles(case, seed)
    pool = PatchPool(0)
    _reserve(pool, [(len(c[1]), (c[2], c[2])) for c in classes])
    layouts, views = [], {}
    for values, pos, n, dx, width, rows in classes:
        slots = _register(pool, pos, n * dx, (n, n))
        _write(pool, slots, (n, n), pool.current_state(0), values)
        grid = np.full(width * rows, -1, dtype=np.int32)
        grid[:len(slots)] = slots
        layouts.append(GridLayout(n, grid.reshape(width, rows)))
        v = _tiles(pool, slots[0], len(slots), (n, n), pool.current_state(0), False)
        views.update({"%d_%s" % (n, q): x for q, x in zip(("h", "hu", "hv"), v)})
    return _stepping(pool, case, layouts, views)


def _refine(case):
    """A patch refines where its cells hold both dry and wet cells or the
    depth jumps between neighbouring cells (of seed 0, for every seed)."""
    n = case["n"]
    fn = _field_fn(case, 0)

    def refine(lev, ij):
        if lev >= case["levels"]:
            return False
        size = 1.0 / (case["px"] * 3 ** (lev - 1))
        c = (np.arange(n) + 0.5) * (size / n)
        h, _ = fn(*np.meshgrid(ij[0] * size + c, ij[1] * size + c, indexing="ij"))
        dry = h == 0.0
        if dry.any() and not dry.all():
            return True
        return bool(max(np.abs(np.diff(h, axis=0)).max(), np.abs(np.diff(h, axis=1)).max())
                    > 0.5)
    return refine


def _prepare_tree(case, seed):
    fn = _field_fn(case, seed)
    pool = PatchPool(0)
    n = case["n"]
    px = case["px"]
    grid = AmrGrid(DeviceBackend(pool), px, px, n, _refine(case), fn,
                   max_level=case["levels"])
    slots = [p.handle for p in grid.leaves]
    first = min(s for lev in grid.levels.values() for s in (p.handle for p in lev.values()))
    count = len(grid.leaves) + len(grid.virtuals)
    all_tiles = _tiles(pool, first, count, (n, n), pool.current_state(0), False)[:3]
    return State(case, pool=pool, grid=grid, tiles=all_tiles,
                 leaves=torch.as_tensor(np.array(slots) - first, device=DEV))


def _prepare_amr(case, seed):
    s = _prepare_tree(case, seed)
    s.amr = BatchedAmr(s.grid)
    return s


def _prepare_lts(case, seed):
    s = _prepare_amr(case, seed)
    s.amr.lts_init()
    return s


def _prepare_calls(case, seed):
    return _prepare_tree(case, seed)


def _regrid_geometry(case):
    side = int(math.ceil(math.sqrt(case["parents"])))
    size = 1.0 / side
    pos = [((k // side) * size, (k % side) * size) for k in range(case["parents"])]
    fine = [(p[0] + a * (size / 3.0), p[1] + c * (size / 3.0)) for p in pos for a in range(3)
            for c in range(3)]
    return pos, fine, size


REGRID_CLOCK = (0.1, 0.004)  # time and step of every leaf at the regrid


def _regrid_values(case, seed):
    """uOld and uNew of the coarse patches (random smooth fields over bumps)
    and b of all three kinds of patch."""
    rng = _rng(case, seed)
    pos, fine, size = _regrid_geometry(case)
    n = (case["n"], case["n"])
    X, Y = torch.broadcast_tensors(*_centres(pos, (size, size), n))
    fields = []
    for base, amp in ((1.2, 0.3), (0.0, 0.2), (0.0, 0.2)) * 2:
        f = torch.full_like(X, base)
        for _ in range(3):
            kx, ky, ph = rng.uniform(2, 40), rng.uniform(2, 40), rng.uniform(0, 6)
            f += amp / 3 * torch.sin(kx * X + ky * Y + ph)
        fields.append(f)
    fn = _dam(rng, 5, 2.0)
    FX, FY = torch.broadcast_tensors(*_centres(fine, (size / 3.0, size / 3.0), n))
    return fields[:3], fields[3:], fn(X, Y, torch)[1], fn(FX, FY, torch)[1]


def _prepare_regrid(case, seed):
    pos, fine, size = _regrid_geometry(case)
    old, new, b, bf = _regrid_values(case, seed)
    n = (case["n"], case["n"])
    pool = PatchPool(0)
    t, dt = REGRID_CLOCK
    _reserve(pool, [(11 * len(pos), n)])
    kw = {"time": t, "timestep_size": dt}
    parents = _register(pool, pos, size, n, level=1, **kw)
    children = _register(pool, fine, size / 3.0, n, level=2, **kw)
    virtual = _register(pool, pos, size, n, level=1, is_virtual=True, **kw)
    cur = pool.current_state(0)
    _write(pool, parents, n, cur, new + [b])
    _write(pool, parents, n, 1 - cur, old + [None])
    _write(pool, children, n, cur, [None] * 3 + [bf])
    _write(pool, virtual, n, cur, [None] * 3 + [b])
    full = (case["n"], case["n"])
    calls = [c for k, p in enumerate(parents) for ch in children[9 * k:9 * k + 9]
             for c in ((full, (0, 0), p, ch, 0, 0, 0), (full, (0, 0), p, ch, 1, 1, 0))]
    pairs = [(ch, v) for k, v in enumerate(virtual) for ch in children[9 * k:9 * k + 9]]
    views = {}
    for name, slots in (("fine", children), ("coarse", virtual)):
        for st, which in (("new", cur), ("old", 1 - cur)):
            v = _tiles(pool, slots[0], len(slots), n, which, False)
            views.update({"%s_%s_%s" % (name, st, q): x for q, x in zip(("h", "hu", "hv"), v)})
    dx = size / case["n"]
    return State(case, pool=pool, backend=DeviceBackend(pool), calls=calls, pairs=pairs,
                 virtual=virtual, views=views, widths=(dx / 3.0, dx))


def _requests(case, seed):
    rng = _rng(case, seed)
    out = []
    for k in range(case["requests"]):
        # the first and last of a burst are the ends of the range
        f = k / max(1, case["requests"] - 1)
        n = math.exp(math.log(case["n_min"]) * (1 - f) + math.log(case["n_max"]) * f)
        n = SERVE_PATCH * max(1, int(round(n / SERVE_PATCH)))
        out.append({"n": n, "centre": (rng.uniform(0.2, 0.8), rng.uniform(0.2, 0.8)),
                    "height": rng.uniform(1.2, 3.0),
                    "hills": [(rng.uniform(0, 1), rng.uniform(0, 1), rng.uniform(0.05, 0.15),
                               rng.uniform(0.0, 0.3)) for _ in range(5)]})
    return out


def _prepare_serve(case, seed):
    pool = PatchPool(0)
    pool.launch_config(fused=2)
    server = Server(pool, max_active=64, keep_completed=True)
    reqs = [make_request(r["n"], SERVE_PATCH, case["end_time"], r["centre"], 0.1, r["height"],
                         1.0, r["hills"]) for r in _requests(case, seed)]
    return State(case, pool=pool, server=server, requests=reqs, kept=[])


# ---- run ----

def run(s):
    kind = s.case["kind"]
    if kind in ("grid", "uneven"):
        if s.case.get("form") == "graph":
            s.pool.graph_replay(s.case["steps"])
        else:
            s.pool.step(s.case["steps"])
        return s.views
    if kind == "amr":
        s.amr.step(s.case["steps"])
        return _leaf_values(s)
    if kind == "lts":
        s.amr.lts_iterations(s.case["steps"], 1e9)
        return _leaf_values(s)
    if kind == "calls":
        for _ in range(s.case["steps"]):
            s.grid.step()
        s.pool.synchronize()
        return _leaf_values(s)
    if kind == "regrid":
        b = s.backend
        flags = s.pool.refinement_flags(0.05, *s.widths)
        b.interpolate_batch(s.calls)
        b.clear_batch(s.virtual)
        b.restrict_batch(s.pairs)
        for v in s.virtual:
            b.post_restrict(v)
        s.pool.synchronize()
        return dict(s.views, flags=flags)
    return _run_serve(s)


def _leaf_values(s):
    return {q: t[s.leaves] for q, t in zip(("h", "hu", "hv"), s.tiles)}


def _run_serve(s):
    for rid in s.kept:  # the results of the last burst have been read
        s.server.release(rid)
    ids = [s.server.submit(r) for r in s.requests]
    results = {}
    while len(results) < len(ids):
        s.server.round(SERVE_ROUND)
        for r in s.server.poll():
            results[r.id] = r
    s.kept = ids
    out = {}
    for k, rid in enumerate(ids):
        slots = s.server.slots(rid)
        state = s.pool.current_state(results[rid].scenario)
        v = _tiles(s.pool, slots[0], len(slots), (SERVE_PATCH, SERVE_PATCH), state, False)
        out.update({"r%d_%s" % (k, q): x for q, x in zip(("h", "hu", "hv"), v)})
    res = [results[rid] for rid in ids]
    out["steps"] = np.array([r.steps for r in res], dtype=np.int64)
    out["digest"] = np.array([r.state_hash for r in res], dtype=np.uint64).view(np.int64)
    out["time"] = np.array([r.time for r in res])
    out["mass"] = np.array([r.mass for r in res])
    return out


# ---- work ----

CELL_BYTES = 56    # read h, hu, hv, b; write h, hu, hv
FWAVE_FLOPS = 180  # two edges of about 70, their speeds' bound, the update
AUG_FLOPS = 420


def _tree_counts(case):
    """Leaves of an adaptive case."""
    refine = _refine(case)
    level = [(i, j) for i in range(case["px"]) for j in range(case["px"])]
    leaves = 0
    for lev in range(1, case["levels"] + 1):
        fine = []
        for ij in level:
            if refine(lev, ij):
                fine += [(3 * ij[0] + a, 3 * ij[1] + c) for a in range(3) for c in range(3)]
            else:
                leaves += 1
        level = fine
    return leaves


def work(case):
    kind = case["kind"]
    if kind == "grid":
        cells = case["px"] * case["py"] * case["nx"] * case["ny"] * case["steps"]
    elif kind == "uneven":
        cells = sum(n * n * c for n, c in _uneven_counts(case).items()) * case["steps"]
    elif kind in ("amr", "calls"):
        cells = _tree_counts(case) * case["n"] ** 2 * case["steps"]
    elif kind == "lts":
        # about an eighth of the leaves advances in an iteration
        cells = _tree_counts(case) * case["n"] ** 2 * case["steps"] / 8
    elif kind == "serve":
        # steps to the end time at about 0.4 dx / 6
        cells = sum(r["n"] ** 2 * math.ceil(case["end_time"] * r["n"] * 6 / 0.4)
                    for r in _requests(case, 0))
    else:
        # coarse: 3 fields x 2 states + b read, 6 written; fine: 6 written by
        # the interpolation and read again by the restriction, b read twice
        # (both kinds of call); h of every patch read by the flags
        area = case["parents"] * case["n"] ** 2
        return {"bytes": 8 * area * (7 + 7 + 9 * 14 + 11), "flops": area * (9 * 2 * 60 + 9 * 40)}
    flops = AUG_FLOPS if case.get("solver", 1) == 2 else FWAVE_FLOPS
    return {"bytes": cells * CELL_BYTES, "flops": cells * flops}


# ---- exact: the same computation on batches of tiles in plain torch ----

def _fwave(hL, hR, qL, qR, bL, bR):
    """Net updates (dhL, dhR, dqL, dqR) and the speed of f-wave edges."""
    lw, rw = hL >= DRY, hR >= DRY
    rd, ld, both = lw & ~rw, ~lw & rw, ~lw & ~rw
    hL, hR = torch.where(ld, hR, hL), torch.where(rd, hL, hR)
    qL, qR = torch.where(ld, -qR, qL), torch.where(rd, -qL, qR)
    bL, bR = torch.where(ld, bR, bL), torch.where(rd, bL, bR)
    one = torch.ones_like(hL)
    hL, hR = torch.where(both, one, hL), torch.where(both, one, hR)
    uL, uR = qL / hL, qR / hR
    sL, sR = hL.sqrt(), hR.sqrt()
    u = (uL * sL + uR * sR) / (sL + sR)
    c = (GRAVITY * 0.5 * (hL + hR)).sqrt()
    s1 = torch.minimum(uL - (GRAVITY * hL).sqrt(), u - c)
    s2 = torch.maximum(uR + (GRAVITY * hR).sqrt(), u + c)
    d0 = qR - qL
    d1 = (qR * uR + 0.5 * GRAVITY * hR * hR) - (qL * uL + 0.5 * GRAVITY * hL * hL) \
        + 0.5 * GRAVITY * (hL + hR) * (bR - bL)
    beta1, beta2 = (s2 * d0 - d1) / (s2 - s1), (d1 - s1 * d0) / (s2 - s1)
    out = [torch.zeros_like(hL) for _ in range(4)]
    for s, f in ((s1, beta1), (s2, beta2)):
        _split(out, s, f, f * s)
    for k, gone in ((0, ld | both), (2, ld | both), (1, rd | both), (3, rd | both)):
        out[k] = torch.where(gone, torch.zeros_like(hL), out[k])
    speed = torch.maximum(s1.abs(), s2.abs())
    return out + [torch.where(both, torch.zeros_like(speed), speed)]


def _split(out, s, fh, fq):
    """One wave of speed s onto the cells left and right of the edge."""
    left = torch.where(s < -ZERO, 1.0, torch.where(s > ZERO, 0.0, 0.5)).to(F64)
    out[0] = out[0] + left * fh
    out[1] = out[1] + (1.0 - left) * fh
    out[2] = out[2] + left * fq
    out[3] = out[3] + (1.0 - left) * fq


def _middle(hL, hR, uL, uR):
    """Middle depth and speeds of the Riemann problem on a flat bottom (two
    rarefactions; two shocks, one Newton step; one of each, one chord step)."""
    g = GRAVITY
    lo, hi = torch.minimum(hL, hR), torch.maximum(hL, hR)
    du = uR - uL
    tiny = lo <= DRY
    slo, shi = torch.where(tiny, 1.0, lo), torch.where(tiny, 1.0, hi)
    sl, sr = torch.where(tiny, 1.0, hL), torch.where(tiny, 1.0, hR)
    cmax = (g * shi).sqrt()
    fmin = du + 2.0 * ((g * slo).sqrt() - cmax)
    fmax = du + (shi - slo) * (0.5 * g * (shi + slo) / (shi * slo)).sqrt()
    cL, cR = (g * sl).sqrt(), (g * sr).sqrt()
    w = torch.clamp(2.0 * (cL + cR) - du, min=0.0)
    h_rr = w * w / (16.0 * g)
    gL, gR = (0.5 * g * (1 / shi + 1 / sl)).sqrt(), (0.5 * g * (1 / shi + 1 / sr)).sqrt()
    f0 = (du + (shi - sl) * gL) + (shi - sr) * gR
    dfdh = gL - g * (shi - sl) / (4 * shi * shi * gL) + gR - g * (shi - sr) / (4 * shi * shi * gR)
    h_ss = (shi.sqrt() - f0 / (2 * shi.sqrt() * dfdh)) ** 2
    h_sr = slo - fmin / torch.where(shi > slo, (fmax - fmin) / (shi - slo), torch.ones_like(slo))
    two_r, two_s = fmin > 0.0, fmax <= 0.0
    hm = torch.where(two_r, h_rr, torch.where(two_s, h_ss, h_sr))
    cm = torch.clamp(g * hm, min=0.0).sqrt()
    safe = torch.where(hm > 0.0, hm, torch.ones_like(hm))
    u1 = uL - (hm - sl) * (0.5 * g * (1 / safe + 1 / sl)).sqrt()
    u2 = uR + (hm - sr) * (0.5 * g * (1 / safe + 1 / sr)).sqrt()
    left = sl > sr
    wl, wr = uL + 2.0 * cL, uR - 2.0 * cR
    s1 = torch.where(two_r, wl - 3.0 * cm, torch.where(
        two_s, u1 - cm, torch.where(left, wl - 3.0 * cm, wr + cm)))
    s2 = torch.where(two_r, wr + 3.0 * cm, torch.where(
        two_s, u2 + cm, torch.where(left, wl - cm, wr + 3.0 * cm)))
    dry = (uR + uL - 2.0 * (g * hR).sqrt()) + 2.0 * (g * hL).sqrt()
    return (torch.where(tiny, torch.zeros_like(hm), hm), torch.where(tiny, dry, s1),
            torch.where(tiny, dry, s2))


def _augmented(hL, hR, qL, qR, bL, bR):
    """The same of augmented Riemann edges (George, J. Comput. Phys. 227)."""
    g, crit = GRAVITY, 1e-6
    zero, one = torch.zeros_like(hL), torch.ones_like(hL)
    lw, rw = hL > DRY, hR > DRY
    both = ~lw & ~rw
    hL, qL = torch.where(lw, hL, zero), torch.where(lw, qL, zero)
    hR, qR = torch.where(rw, hR, zero), torch.where(rw, qR, zero)
    uL = torch.where(lw, qL / torch.where(lw, hL, one), zero)
    uR = torch.where(rw, qR / torch.where(rw, hR, one), zero)
    pL, pR = 0.5 * g * hL * hL + qL * uL, 0.5 * g * hR * hR + qR * uR
    rd, ld = lw & ~rw, ~lw & rw
    reach_l = torch.maximum(hL, _middle(hL, hL, uL, -uL)[0]) + bL
    reach_r = torch.maximum(hR, _middle(hR, hR, -uR, uR)[0]) + bR
    wall_r, wall_l = rd & (reach_l < bR), ld & (reach_r < bL)
    bR = torch.where(rd & ~wall_r & (hL + bL < bR), hL + bL, bR)
    bL = torch.where(ld & ~wall_l & (hR + bR < bL), hR + bR, bL)
    hR, qR, bR, pR, uR = (torch.where(wall_r, a, c) for a, c in (
        (hL, hR), (-qL, qR), (bL, bR), (pL, pR), (-uL, uR)))
    hL, qL, bL, pL, uL = (torch.where(wall_l, a, c) for a, c in (
        (hR, hL), (-qR, qL), (bR, bL), (pR, pL), (-uR, uL)))
    hL, hR = torch.where(both, one, hL), torch.where(both, one, hR)
    w0 = torch.where(wall_l, zero, one)
    w2 = torch.where(wall_r, zero, one)
    w1 = w0 * w2
    cL, cR = (g * hL).sqrt(), (g * hR).sqrt()
    uh = (cL * uL + cR * uR) / (cR + cL)
    ch = (g * 0.5 * (hR + hL)).sqrt()
    _, s1m, s2m = _middle(hL, hR, uL, uR)
    l1 = torch.minimum(torch.minimum(uL - cL, uh - ch), s2m)
    l3 = torch.maximum(torch.maximum(uR + cR, uh + ch), s1m)
    l2 = 0.5 * (l1 + l3)
    db, hbar = bR - bL, 0.5 * (hL + hR)
    star = torch.clamp((qL - qR + l3 * hR - l1 * hL) / (l3 - l1), min=0.0)
    sbar = 0.25 * (uL + uR) ** 2 - g * hbar
    stil = torch.clamp(uL * uR, min=0.0) - g * hbar
    sonic = (sbar.abs() <= crit) | (sbar * stil <= crit) | (sbar * l1 * l3 <= crit) \
        | (torch.minimum(l1.abs(), l3.abs()) < crit) | ((l1 < 0) & (s1m > 0)) \
        | ((l3 > 0) & (s2m < 0)) | ((uL + cL) * (uR + cR) < 0) | ((uL - cL) * (uR - cR) < 0)
    sden = torch.where(sonic, one, sbar)
    ddh = torch.where(sonic, -db, db * g * hbar / sden)
    up, lo = star * (l3 - l1) / l3, star * (l3 - l1) / l1
    sub = (l1 < -crit) & (l3 > crit)
    right, left = ~sub & (l1 >= crit), ~sub & ~(l1 >= crit) & (l3 <= -crit)
    ddh = torch.where(sub, torch.maximum(torch.minimum(ddh, up), lo), torch.where(
        right, torch.maximum(torch.minimum(ddh, lo), -hL), torch.where(
            left, torch.maximum(torch.minimum(ddh, hR), up), ddh)))
    ddp = torch.where(sonic, -g * hbar * db, -db * g * hbar * stil / sden)
    ddp = torch.minimum(ddp, g * torch.maximum(-hL * db, -hR * db))
    ddp = torch.maximum(ddp, g * torch.minimum(-hL * db, -hR * db))
    d0, d1, d2 = hR - hL - ddh, qR - qL, pR - pL - ddp
    beta0 = (l3 * d0 - d1) / (l3 - l1)
    beta2 = (d1 - l1 * d0) / (l3 - l1)
    beta1 = d2 - beta0 * l1 * l1 - beta2 * l3 * l3
    out = [zero, zero, zero, zero]
    for s, w, fh, fq in ((l1, w0, beta0 * l1, beta0 * l1 * l1), (l2, w1, zero, beta1),
                         (l3, w2, beta2 * l3, beta2 * l3 * l3)):
        _split(out, s * w, fh * w, fq * w)
    out = [torch.where(both, zero, x) for x in out]
    speed = torch.maximum(torch.maximum((l1 * w0).abs(), (l2 * w1).abs()), (l3 * w2).abs())
    return out + [torch.where(both, zero, speed)]


def _net(u, solver, spacing):
    """Net updates of the interior cells of filled tiles u = (h, hu, hv, b)
    and every tile's largest edge speed."""
    edge = _augmented if solver == 2 else _fwave
    h, hu, hv, b = u
    xl, xr = (slice(None), slice(0, -1), slice(1, -1)), (slice(None), slice(1, None), slice(1, -1))
    yl, yr = (slice(None), slice(1, -1), slice(0, -1)), (slice(None), slice(1, -1), slice(1, None))
    aL, aR, cL, cR, s = edge(h[xl], h[xr], hu[xl], hu[xr], b[xl], b[xr])
    top = s.amax((1, 2))
    dx, dy = spacing
    nh = (aR[:, :-1] + aL[:, 1:]) / dx
    nhu = (cR[:, :-1] + cL[:, 1:]) / dx
    aL, aR, cL, cR, s = edge(h[yl], h[yr], hv[yl], hv[yr], b[yl], b[yr])
    nh = nh + (aR[:, :, :-1] + aL[:, :, 1:]) / dy
    nhv = (cR[:, :, :-1] + cL[:, :, 1:]) / dy
    return (nh, nhu, nhv), torch.maximum(top, s.amax((1, 2)))


def _cfl(top, spacing):
    t = CFL * min(spacing) / torch.where(top > 1e-5, top, torch.ones_like(top))
    return torch.where(top > 1e-5, t, torch.full_like(t, 1.7976931348623157e308))


def _updated(u, net, dt):
    h, hu, hv = (q[:, 1:-1, 1:-1] - dt * f for q, f in zip(u[:3], net))
    still = h < 0.1
    return (torch.clamp(h, min=0.0), torch.where(still, torch.zeros_like(hu), hu),
            torch.where(still, torch.zeros_like(hv), hv))


def _walls(u, sides):
    """Reflective walls of the tiles that `sides` ((4, tiles) truth values:
    x-, x+, y-, y+) marks."""
    for k, (ghost, own, flip) in enumerate((((0,), (1,), 1), ((-1,), (-2,), 1),
                                            ((slice(None), 0), (slice(None), 1), 2),
                                            ((slice(None), -1), (slice(None), -2), 2))):
        for q in range(3):
            v = u[q]
            g, o = (slice(None),) + ghost, (slice(None),) + own
            v[g] = torch.where(sides[k][:, None], -v[o] if q == flip else v[o], v[g])


class _Uniform:
    """Tiles of one px x py grid (missing ones at the end)."""

    def __init__(self, values, px, py, spacing, solver):
        self.u = [v.clone() for v in values]
        self.spacing, self.solver = spacing, solver
        k = torch.arange(px * py, device=DEV)
        i, j = k // py, k % py
        count = self.u[0].shape[0]
        self.nb = []
        for di, dj in ((-1, 0), (1, 0), (0, -1), (0, 1)):
            a, c = i + di, j + dj
            q = torch.where((a >= 0) & (a < px) & (c >= 0) & (c < py), a * py + c, -1)
            self.nb.append(torch.where(q < count, q, -1)[:count])

    def net(self):
        cut = (((0,), (-2,)), ((-1,), (1,)), ((slice(None), 0), (slice(None), -2)),
               ((slice(None), -1), (slice(None), 1)))
        for q, (ghost, own) in zip(self.nb, cut):
            g, o = (slice(None),) + ghost, (slice(None),) + own
            for v in self.u[:3]:
                v[g] = torch.where((q >= 0)[:, None], v[o][q.clamp(min=0)], v[g])
        _walls(self.u, [q < 0 for q in self.nb])
        return _net(self.u, self.solver, self.spacing)

    def update(self, net, dt):
        for v, x in zip(self.u[:3], _updated(self.u, net, dt)):
            v[:, 1:-1, 1:-1] = x

    def interior(self):
        return [v[:, 1:-1, 1:-1] for v in self.u[:3]]


def _march(grids, steps=None, end=math.inf):
    """Global steps of several grids; returns the steps taken and the time."""
    t = taken = 0
    while (steps is None or taken < steps) and end - t > EPS:
        nets = [g.net() for g in grids]
        dt = min(min(float(_cfl(top, g.spacing).min()) for g, (_, top) in zip(grids, nets)),
                 end - t)
        for g, (net, _) in zip(grids, nets):
            g.update(net, dt)
        t += dt
        taken += 1
    return taken, t


class _Tree:
    """An adaptive grid: per level the leaf tiles with their own clocks, and
    composites over the whole domain for what lies across their faces."""

    def __init__(self, case, seed):
        fn = _field_fn(case, seed)
        refine = _refine(case)
        self.n, self.px = case["n"], case["px"]
        n = self.n
        self.levels = []
        cells = [(i, j) for i in range(self.px) for j in range(self.px)]
        for lev in range(1, case["levels"] + 1):
            side = self.px * 3 ** (lev - 1)
            leaf = torch.zeros((side, side), dtype=torch.bool)
            virt = torch.zeros_like(leaf)
            fine = []
            for ij in cells:
                if refine(lev, ij):
                    virt[ij] = True
                    fine += [(3 * ij[0] + a, 3 * ij[1] + c) for a in range(3) for c in range(3)]
                else:
                    leaf[ij] = True
            # the grid's own order: level by level, children parent by parent
            ids = torch.tensor([ij for ij in cells if leaf[ij]], device=DEV).reshape(-1, 2)
            size = 1.0 / side
            X, Y = torch.broadcast_tensors(*_centres((ids.to(F64) * size).cpu().numpy(),
                                                     (size, size), (n, n)))
            h, b = fn(X, Y, torch)
            u = [h[:, 1:-1, 1:-1].clone()] + [torch.zeros_like(h[:, 1:-1, 1:-1])
                                              for _ in range(2)]
            zero = torch.zeros(len(ids), dtype=F64, device=DEV)
            self.levels.append({"side": side, "leaf": leaf.to(DEV), "virt": virt.to(DEV),
                                "ids": ids, "new": u, "old": [torch.zeros_like(x) for x in u],
                                "b": b, "t": zero, "dt": zero.clone(),
                                "spacing": (size / n, size / n)})
            cells = fine

    def _paste(self, lv, tiles):
        n, side = self.n, lv["side"]
        out = torch.zeros((side, side, n, n), dtype=F64, device=DEV)
        out[lv["ids"][:, 0], lv["ids"][:, 1]] = tiles
        return out.permute(0, 2, 1, 3).reshape(side * n, side * n)

    def _mask(self, m):
        return m.repeat_interleave(self.n, 0).repeat_interleave(self.n, 1)

    def _bilinear(self, f, side, factor):
        """Dense field of a level at the cells `factor` finer, linear inside
        each patch (extrapolated to its border)."""
        n = self.n
        u = (torch.arange(n * factor, dtype=F64, device=DEV) + 0.5) / factor - 0.5
        i0 = u.floor().long().clamp(0, n - 2)
        w = u - i0
        at = (torch.arange(side, device=DEV)[:, None] * n + i0[None, :]).reshape(-1)
        w = w.repeat(side)
        f = f[at] * (1 - w)[:, None] + f[at + 1] * w[:, None]
        return f[:, at] * (1 - w)[None, :] + f[:, at + 1] * w[None, :]

    def _composites(self):
        """Per level (A, B) of h + b, hu, hv over the domain: the value at time
        T is A + B T (leaves between their two states, virtual patches as the
        mean of what is below, elsewhere the coarser leaf's interpolation)."""
        dense = []
        for lv in self.levels:
            moving = (lv["dt"] > EPS)[:, None, None]
            step = torch.where(moving, lv["dt"][:, None, None], 1.0)
            ab = []
            for q in range(3):
                new, old = lv["new"][q], lv["old"][q]
                if q == 0:
                    bb = lv["b"][:, 1:-1, 1:-1]
                    new, old = new + bb, old + bb
                slope = torch.where(moving, (new - old) / step, torch.zeros_like(new))
                const = torch.where(moving, old - slope * lv["t"][:, None, None], new)
                ab += [self._paste(lv, const), self._paste(lv, slope)]
            dense.append(ab)
        for k in range(len(dense) - 2, -1, -1):
            m = self._mask(self.levels[k]["virt"])
            for c in range(6):
                mean = torch.nn.functional.avg_pool2d(dense[k + 1][c][None, None], 3)[0, 0]
                dense[k][c] = torch.where(m, mean, dense[k][c])
        leaf_only = [[x.clone() for x in d] for d in dense]
        for k in range(1, len(dense)):
            for j in range(k):
                f = 3 ** (k - j)
                m = self._mask(self.levels[j]["leaf"]).repeat_interleave(f, 0) \
                    .repeat_interleave(f, 1)
                for c in range(6):
                    fine = self._bilinear(leaf_only[j][c], self.levels[j]["side"], f)
                    dense[k][c] = torch.where(m, fine, dense[k][c])
        return dense

    def _filled(self, lv, ab):
        """Tiles of a level's leaves with their ghost layers at the end of
        each leaf's interval."""
        n = self.n
        at = torch.arange(-1, n + 1, device=DEV)
        top = lv["side"] * n - 1
        ii = (lv["ids"][:, 0, None] * n + at).clamp(0, top)
        jj = (lv["ids"][:, 1, None] * n + at).clamp(0, top)
        when = (lv["t"] + lv["dt"])[:, None, None]
        u = []
        for q in range(3):
            v = ab[2 * q][ii[:, :, None], jj[:, None, :]] \
                + ab[2 * q + 1][ii[:, :, None], jj[:, None, :]] * when
            if q == 0:
                v = v - lv["b"]
            v[:, 1:-1, 1:-1] = lv["new"][q]
            u.append(v)
        i, j = lv["ids"][:, 0], lv["ids"][:, 1]
        _walls(u, [i == 0, i == lv["side"] - 1, j == 0, j == lv["side"] - 1])
        return u + [lv["b"]]

    def _advancing(self):
        """Local time stepping: leaves no neighbour (face or corner) holds back."""
        ends = []
        for lv in self.levels:
            e = torch.full((lv["side"], lv["side"]), math.inf, dtype=F64, device=DEV)
            e[lv["ids"][:, 0], lv["ids"][:, 1]] = lv["t"] + lv["dt"]
            ends.append(e)
        for k in range(len(ends) - 2, -1, -1):
            low = -torch.nn.functional.max_pool2d(-ends[k + 1][None, None], 3)[0, 0]
            ends[k] = torch.where(self.levels[k]["virt"], low, ends[k])
        for k in range(1, len(ends)):
            lv = self.levels[k]
            coarse = ends[k - 1].repeat_interleave(3, 0).repeat_interleave(3, 1)
            ends[k] = torch.where(lv["leaf"] | lv["virt"], ends[k], coarse)
        out = []
        for lv, e in zip(self.levels, ends):
            pad = torch.nn.functional.pad(-e[None, None], (1, 1, 1, 1), value=-math.inf)
            low = -torch.nn.functional.max_pool2d(pad, 3, 1)[0, 0]
            i, j = lv["ids"][:, 0], lv["ids"][:, 1]
            out.append(~(e[i, j] - low[i, j] > EPS))
        return out

    def step(self, local):
        dense = self._composites()
        go = self._advancing() if local else None
        work_ = []
        for lv, ab in zip(self.levels, dense):
            if not len(lv["ids"]):
                work_.append(None)
                continue
            u = self._filled(lv, ab)
            net, top = _net(u, 1, lv["spacing"])
            work_.append((u, net, _cfl(top, lv["spacing"])))
        whole = min(float(w[2].min()) for w in work_ if w is not None)
        for k, (lv, w) in enumerate(zip(self.levels, work_)):
            if w is None:
                continue
            u, net, cfl = w
            dt = cfl if local else torch.full_like(cfl, whole)
            m = go[k] if local else torch.ones_like(cfl, dtype=torch.bool)
            new = _updated(u, net, dt[:, None, None])
            for q in range(3):
                lv["old"][q] = torch.where(m[:, None, None], lv["new"][q], lv["old"][q])
                lv["new"][q] = torch.where(m[:, None, None], new[q], lv["new"][q])
            lv["t"] = torch.where(m, lv["t"] + lv["dt"], lv["t"])
            lv["dt"] = torch.where(m, dt, lv["dt"])

    def leaves(self):
        return [torch.cat([lv["new"][q] for lv in self.levels]) for q in range(3)]


def _exact_regrid(case, seed):
    old, new, b, bf = _regrid_values(case, seed)
    n = case["n"]
    t, dt = REGRID_CLOCK
    # children of parent k at (a, c): linear inside the parent
    u = (torch.arange(3 * n, dtype=F64, device=DEV) + 0.5) / 3 - 0.5
    i0 = u.floor().long().clamp(0, n - 2)
    w = u - i0
    out, mean = {}, {}
    for name, fields in (("new", new), ("old", old)):
        for q, f in zip(("h", "hu", "hv"), fields):
            f = f[:, 1:-1, 1:-1] + (b[:, 1:-1, 1:-1] if q == "h" else 0.0)
            f = f[:, i0] * (1 - w)[None, :, None] + f[:, i0 + 1] * w[None, :, None]
            f = f[:, :, i0] * (1 - w) + f[:, :, i0 + 1] * w
            mean[name, q] = torch.nn.functional.avg_pool2d(f[:, None], 3)[:, 0]
            f = f.reshape(-1, 3, n, 3, n).permute(0, 1, 3, 2, 4).reshape(-1, n, n)
            out["fine_%s_%s" % (name, q)] = f - (bf[:, 1:-1, 1:-1] if q == "h" else 0.0)
    # restriction to the values at times 0 and 1
    for q in ("h", "hu", "hv"):
        slope = (mean["new", q] - mean["old", q]) / dt
        for name, when in (("old", 0.0), ("new", 1.0)):
            v = mean["old", q] + slope * (when - t)
            out["coarse_%s_%s" % (name, q)] = v - (b[:, 1:-1, 1:-1] if q == "h" else 0.0)
    return dict(out, flags=None)


def _exact_serve(case, seed):
    out = {"steps": None, "digest": None}
    times, masses = [], []
    for k, r in enumerate(_requests(case, seed)):
        p = r["n"] // SERVE_PATCH
        size = 1.0 / p
        pos = [(i * size, j * size) for i in range(p) for j in range(p)]
        X, Y = torch.broadcast_tensors(*_centres(pos, (size, size), (SERVE_PATCH, SERVE_PATCH)))
        near = (X - r["centre"][0]) ** 2 + (Y - r["centre"][1]) ** 2 <= 0.1 ** 2
        b = torch.zeros_like(X)
        h = torch.where(near, b + r["height"], b + 1.0)
        for x, y, s, a in r["hills"]:
            b = b + a * torch.exp(-((X - x) ** 2 + (Y - y) ** 2) / (s * s))
        z = torch.zeros_like(h)
        g = _Uniform([h, z, z, b], p, p, (1.0 / r["n"], 1.0 / r["n"]), 1)
        _, t = _march([g], end=case["end_time"])
        for q, v in zip(("h", "hu", "hv"), g.interior()):
            out["r%d_%s" % (k, q)] = v
        times.append(t)
        masses.append(float(g.interior()[0].sum()) / r["n"] ** 2)
    return dict(out, time=np.array(times), mass=np.array(masses))


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        values, _, size, n = _grid_tiles(case, seed)
        g = _Uniform(values, case["px"], case["py"], (size[0] / n[0], size[1] / n[1]),
                     case["solver"])
        _march([g], case["steps"])
        return dict(zip(("h", "hu", "hv"), g.interior()))
    if kind == "uneven":
        grids = [(n, _Uniform(v, width, rows, (dx, dx), 1))
                 for v, _, n, dx, width, rows in _uneven_tiles(case, seed)]
        _march([g for _, g in grids], case["steps"])
        return {"%d_%s" % (n, q): v for n, g in grids
                for q, v in zip(("h", "hu", "hv"), g.interior())}
    if kind in ("amr", "lts", "calls"):
        tree = _Tree(case, seed)
        for _ in range(case["steps"]):
            tree.step(kind == "lts")
        return dict(zip(("h", "hu", "hv"), tree.leaves()))
    if kind == "regrid":
        return _exact_regrid(case, seed)
    return _exact_serve(case, seed)

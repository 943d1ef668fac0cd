"""Steps on short row segments against the row march: the same grids stepped
with automatic row segments (small grids run on segments of at most 1, 2 or 4
rows) and with whole patches (row_segments = 1), bitwise: state, clocks and
the patches' own estimates.  The operations and their order are the same, so
there is no tolerance."""
import math

import numpy as np
import pytest

from peanoclaw_amd.pool import PatchPool, make_description
from peanoclaw_amd.scenarios import GridLayout, Workload

pytestmark = pytest.mark.gpu


def _fill(pool, layouts, scenario, nx, ny, px, py, seed, dry, hole=None, end=math.inf):
    rng = np.random.default_rng(seed)
    grid = -np.ones((px, py), dtype=np.int32)
    for i in range(px):
        for j in range(py):
            if (i, j) == hole:
                continue
            s = pool.register(make_description((i * nx / 64, j * ny / 64), (nx / 64, ny / 64), nx,
                                               ny=ny, scenario=scenario))
            h = rng.uniform(0.5, 2.0, (nx, ny))
            if dry:
                h = np.where(rng.uniform(0, 1, (nx, ny)) < 0.3, 0.0, h)
            m = rng.uniform(-4.0, 4.0, (2, nx, ny)) * h  # some edges supersonic
            pool.upload(s, unew=np.stack([h, m[0], m[1]]),
                        b=rng.uniform(-0.2, 0.2, (nx + 2, ny + 2)))
            grid[i, j] = s
    pool.scenario_set(scenario, 0.0, 0.0, end)
    layouts.append(GridLayout(nx, grid, ny))


def _run(sizes, solver, fused, segments, dry, tile, steps, ends=None):
    out = []
    with PatchPool(0) as pool:
        layouts = []
        for k, (nx, ny, px, py) in enumerate(sizes):
            _fill(pool, layouts, k, nx, ny, px, py, 7 + k, dry,
                  hole=(0, 0) if px * py > 4 else None, end=ends[k] if ends else math.inf)
        wl = Workload(pool, layouts, 0, 0, [])
        wl.build_ghost_table(fused_sides=not tile)
        pool.wave_propagation_solver(solver)
        pool.launch_config(fused=fused)
        pool.row_segments(segments)
        pool.step(1)
        pool.graph_capture()
        pool.graph_replay(steps - 1)
        for k, lay in enumerate(layouts):
            out.append(np.array(pool.scenario_get(k)))
            for s in lay.slot_of.ravel():
                if s >= 0:
                    out.append(pool.download(int(s))[0])
                    out.append(np.array(pool.description(int(s)).estimated_next_timestep_size))
    return out


def _equal(*args, **kw):
    a, b = _run(*args[:3], 0, *args[3:], **kw), _run(*args[:3], 1, *args[3:], **kw)
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


# rows below, at and above the segment lengths; columns around the lane groups
@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 5), (4, 64), (5, 8), (8, 9), (9, 33), (16, 16),
                                   (33, 3), (64, 63), (64, 64)])
@pytest.mark.parametrize("solver", [1, 2])
def test_sizes(nx, ny, solver):
    _equal([(nx, ny, 3, 2)], solver, 0, False, False, 4)


@pytest.mark.parametrize("solver", [1, 2])
@pytest.mark.parametrize("fused", [1, 2])
def test_dry_cells_modes_and_several_scenarios(solver, fused):
    # three sizes in three scenarios; the second ends early
    _equal([(16, 16, 3, 3), (7, 12, 2, 2), (64, 20, 1, 2)], solver, fused, True, False, 6,
           ends=[math.inf, 1e-3, math.inf])


@pytest.mark.parametrize("solver", [1, 2])
def test_tile_ghosts(solver):
    _equal([(8, 16, 3, 3)], solver, 0, True, True, 5)


# enough patches for segments of 4 rows (f-wave) and of 2 rows (augmented)
@pytest.mark.parametrize("solver", [1, 2])
def test_longer_segments(solver):
    _equal([(63, 40, 8, 7)], solver, 2, True, False, 4)


# march steps whose whole patches would leave SIMDs idle are split (here into
# four): the same bits as whole patches
def test_split_march():
    def run(segments):
        with PatchPool(0) as pool:
            layouts = []
            rng = np.random.default_rng(3)
            px = py = 42
            grid = -np.ones((px, py), dtype=np.int32)
            tile = 66 * 80
            pool.reserve(px * py * (tile + 16))
            for k in range(px * py):
                i, j = divmod(k, py)
                grid[i, j] = pool.register(make_description((i, j), 1.0, 64))
            o = [pool.offset(int(s)) for s in grid.ravel()]
            cells = o[-1] + tile - o[0]
            f = [rng.uniform(0.5, 2.0, cells) * a for a in (1.0, 0.3, 0.3, 0.1)]
            pool.copy_fields(True, 0, o[0], *f)
            layouts.append(GridLayout(64, grid))
            wl = Workload(pool, layouts, 0, 0, [])
            wl.build_ghost_table()
            pool.scenario_set(0, 0.0, 0.0, math.inf)
            pool.launch_config(fused=2)
            pool.row_segments(segments)
            pool.step(3)
            out = [np.empty(cells) for _ in range(3)]
            pool.copy_fields(False, 1, o[0], *out)
            out = [a[:px * py * tile - 80].reshape(-1)[:(px * py - 1) * tile]
                   .reshape(-1, 66, 80)[:, 1:-1, 1:65] for a in out]
            return out, pool.scenario_get(0)
    (a, ta), (b, tb) = run(0), run(1)
    assert ta == tb
    for x, y in zip(a, b):
        assert np.array_equal(x, y)

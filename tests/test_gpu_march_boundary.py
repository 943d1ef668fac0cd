"""The boundary pass and the dt stage of the row march with pruned speeds,
against the march with a separate exact speed pass (fused = 0), bitwise: state
and clocks.  dt is the same exact minimum in both, so there is no tolerance."""
import math

import numpy as np
import pytest

from peanoclaw_amd.pool import PatchPool, make_description, tile_stride
from peanoclaw_amd.scenarios import GridLayout, Workload

pytestmark = pytest.mark.gpu

# ghost edges around the lanes a patch gets (8, 16, 32, 64 lanes, up to 4 edges
# each), one patch alone, holes, rectangles; segments add seams to the list
SIZES = [(2, 2, 3, 3), (8, 8, 4, 3), (9, 8, 3, 4), (16, 17, 4, 4), (17, 31, 2, 3), (32, 32, 3, 3),
         (33, 40, 3, 2), (64, 64, 3, 3), (64, 5, 2, 2), (5, 64, 1, 1)]


def _run(fused, segments, slack, scenarios, tile):
    rng = np.random.default_rng(11)
    out = []
    with PatchPool(0) as pool:
        layouts = []
        for k, (nx, ny, px, py) in enumerate(SIZES):
            grid = -np.ones((px, py), dtype=np.int32)
            for i in range(px):
                for j in range(py):
                    if (i, j) == (1, 1):
                        continue
                    s = pool.register(make_description((i, j), (nx / 64, ny / 64), nx, ny=ny,
                                                       scenario=k % scenarios))
                    h = rng.uniform(0.5, 2.0, (nx, ny))
                    m = rng.uniform(-1.0, 1.0, (2, nx, ny)) * h
                    pool.upload(s, unew=np.stack([h, m[0], m[1]]),
                                b=rng.uniform(-0.2, 0.2, (nx + 2, ny + 2)))
                    grid[i, j] = s
            layouts.append(GridLayout(nx, grid, ny))
        for k in range(scenarios):
            pool.scenario_set(k, 0.0, 0.0, math.inf)
        wl = Workload(pool, layouts, 0, 0, [])
        wl.build_ghost_table(fused_sides=not tile)
        pool.launch_config(fused=fused)
        pool.prune_slack(slack)
        pool.row_segments(segments)
        pool.step(2)
        pool.graph_capture()
        pool.graph_replay(3)
        pool.step(1)
        out += [np.array(pool.scenario_get(k)) for k in range(scenarios)]
        for lay in layouts:
            out += [pool.download(int(s))[0] for s in lay.slot_of.ravel() if s >= 0]
    return out


# slack 0.5: no minimum is accepted, every step takes the exact fallback
@pytest.mark.parametrize("fused,slack", [(1, 1.03125), (2, 1.03125), (2, 0.5)])
@pytest.mark.parametrize("scenarios", [1, 3])
@pytest.mark.parametrize("segments", [1, 4])
def test_against_separate_speed_pass(fused, slack, scenarios, segments):
    a = _run(fused, segments, slack, scenarios, False)
    b = _run(0, 1, 1.03125, scenarios, False)
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


# enough patches that a lane takes 4 edges and a workgroup 8 wavefronts, and
# that the dt stage's workgroups read more than 64 minima
@pytest.mark.parametrize("slack", [1.03125, 0.5])
def test_many_patches(slack):
    def run(fused):
        with PatchPool(0) as pool:
            rng = np.random.default_rng(5)
            px, py, n = 190, 181, 8
            slots = [pool.register(make_description(divmod(k, py), 1.0, n))
                     for k in range(px * py)]
            o = [pool.offset(s) for s in slots]
            cells = o[-1] + (n + 2) * tile_stride(n) - o[0]
            f = [rng.uniform(0.5, 2.0, cells) * a for a in (1.0, 0.3, 0.3, 0.1)]
            pool.copy_fields(True, 0, o[0], *f)
            wl = Workload(pool, [GridLayout(n, np.array(slots, np.int32).reshape(px, py))], 0, 0, [])
            wl.build_ghost_table()
            pool.scenario_set(0, 0.0, 0.0, math.inf)
            pool.launch_config(fused=fused)
            pool.prune_slack(slack)
            pool.row_segments(1)
            pool.step(3)
            return pool.scenario_get(0), [pool.download(s)[0] for s in slots[::211]]
    (ta, a), (tb, b) = run(2), run(0)
    assert ta == tb
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


# 4356 row segments: on segments with fused = 0 and 1, marched with fused = 2;
# changing the mode between steps changes the path, not the bits
def test_mode_changes_the_path():
    def run(segments):
        with PatchPool(0) as pool:
            rng = np.random.default_rng(9)
            p, n = 33, 32
            slots = [pool.register(make_description(divmod(k, p), 1.0, n)) for k in range(p * p)]
            o = [pool.offset(s) for s in slots]
            cells = o[-1] + (n + 2) * tile_stride(n) - o[0]
            pool.copy_fields(True, 0, o[0], *[rng.uniform(0.5, 2.0, cells) * a
                                              for a in (1.0, 0.3, 0.3, 0.1)])
            wl = Workload(pool, [GridLayout(n, np.array(slots, np.int32).reshape(p, p))], 0, 0, [])
            wl.build_ghost_table()
            pool.scenario_set(0, 0.0, 0.0, math.inf)
            pool.row_segments(segments)
            clocks = []
            for fused in (0, 2, 1, 2, 0):
                pool.launch_config(fused=fused)
                pool.step(2)
                clocks.append(pool.scenario_get(0))
                pool.step_per_patch(1) if fused == 2 else pool.step(1)
            return clocks, [pool.download(s)[0] for s in slots[::31]]
    (ta, a), (tb, b) = run(0), run(1)
    assert ta == tb
    for x, y in zip(a, b):
        assert np.array_equal(x, y)

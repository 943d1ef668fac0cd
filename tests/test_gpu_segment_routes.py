"""Steps on short row segments against the row march (row_segments = 1),
bitwise, where many scenarios or many patches decide the route: state, clocks
and the patches' own estimates."""
import math

import numpy as np
import pytest

from peanoclaw_amd.pool import PatchPool, make_description, tile_stride
from peanoclaw_amd.scenarios import GridLayout, Workload

pytestmark = pytest.mark.gpu


# more scenarios than one workgroup advances: numbers around its four
# wavefronts, some scenarios ending early, one without patches
@pytest.mark.parametrize("scenarios", [4, 5, 70])
@pytest.mark.parametrize("solver", [1, 2])
@pytest.mark.parametrize("fused", [0, 2])
def test_many_scenarios(scenarios, solver, fused):
    def run(segments):
        with PatchPool(0) as pool:
            rng = np.random.default_rng(scenarios)
            layouts = []
            for k in range(scenarios):
                if k == 2:
                    continue
                n, px = (8, 16, 12)[k % 3], 1 + k % 2
                grid = np.zeros((px, px), dtype=np.int32)
                for i in range(px):
                    for j in range(px):
                        s = pool.register(make_description((i, j), 1.0, n, scenario=k))
                        h = rng.uniform(0.5, 2.0, (n, n))
                        m = rng.uniform(-1.0, 1.0, (2, n, n)) * h
                        pool.upload(s, unew=np.stack([h, m[0], m[1]]),
                                    b=rng.uniform(-0.2, 0.2, (n + 2, n + 2)))
                        grid[i, j] = s
                pool.scenario_set(k, 0.0, 0.0, 0.01 if k % 5 == 0 else math.inf)
                layouts.append(GridLayout(n, grid))
            Workload(pool, layouts, 0, 0, []).build_ghost_table()
            pool.wave_propagation_solver(solver)
            pool.launch_config(fused=fused)
            pool.row_segments(segments)
            pool.step(4)
            slots = [int(s) for lay in layouts for s in lay.slot_of.ravel()]
            out = [np.array(pool.scenario_get(k)) for k in range(scenarios)]
            out += [pool.download(s)[0] for s in slots]
            return out + [np.array(pool.description(s).estimated_next_timestep_size)
                          for s in slots]
    for x, y in zip(run(0), run(1)):
        assert np.array_equal(x, y)


# the augmented solver on segments of 4 rows: more wavefronts at 2 rows than
# its limit (33 x 33 patches of 8 x 64: 4356)
@pytest.mark.parametrize("dry", [False, True])
def test_augmented_four_rows(dry):
    def run(segments):
        with PatchPool(0) as pool:
            rng = np.random.default_rng(17)
            p, nx, ny = 33, 8, 64
            slots = [pool.register(make_description(divmod(k, p), (nx / 64, ny / 64), nx, ny=ny))
                     for k in range(p * p)]
            o = [pool.offset(s) for s in slots]
            cells = o[-1] + (nx + 2) * tile_stride(ny) - o[0]
            f = [rng.uniform(0.5, 2.0, cells) * a for a in (1.0, 0.3, 0.3, 0.1)]
            if dry:
                f[0][rng.uniform(0.0, 1.0, cells) < 0.2] = 0.0
            pool.copy_fields(True, 0, o[0], *f)
            grid = np.array(slots, np.int32).reshape(p, p)
            Workload(pool, [GridLayout(nx, grid, ny)], 0, 0, []).build_ghost_table()
            pool.scenario_set(0, 0.0, 0.0, math.inf)
            pool.wave_propagation_solver(2)
            pool.row_segments(segments)
            pool.step(3)
            return ([np.array(pool.scenario_get(0))] + [pool.download(s)[0] for s in slots[::7]] +
                    [np.array(pool.description(s).estimated_next_timestep_size)
                     for s in slots[::7]])
    for x, y in zip(run(0), run(1)):
        assert np.array_equal(x, y)

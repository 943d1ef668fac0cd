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

"""Changes of launch mode and calls without a step between batched steps,
bitwise against one mode throughout: the modes differ in how they find the
same speeds."""
import math

import numpy as np
import pytest

from peanoclaw_amd.pool import PatchPool, make_description
from peanoclaw_amd.scenarios import GridLayout, Workload

pytestmark = pytest.mark.gpu


def _pool(n, px, py):
    pool = PatchPool(0)
    rng = np.random.default_rng(n)
    grid = -np.ones((px, py), dtype=np.int32)
    for i in range(px):
        for j in range(py):
            s = pool.register(make_description((i, j), 1.0, n))
            h = rng.uniform(0.5, 2.0, (n, n))
            m = rng.uniform(-1.0, 1.0, (2, n, n)) * h
            pool.upload(s, unew=np.stack([h, m[0], m[1]]),
                        b=rng.uniform(-0.2, 0.2, (n + 2, n + 2)))
            grid[i, j] = s
    pool.scenario_set(0, 0.0, 0.0, math.inf)
    Workload(pool, [GridLayout(n, grid)], 0, 0, []).build_ghost_table()
    return pool, [int(s) for s in grid.ravel()]


# slack below 1: the pruned interior speeds are mostly missing and every
# pruned step takes the exact fallback, so another mode must not use them
@pytest.mark.parametrize("n", [8, 33, 64])
@pytest.mark.parametrize("slack", [0.5, 1.03125])
def test_pruned_to_exact(n, slack):
    def run(modes):
        pool, slots = _pool(n, 3, 4)
        with pool:
            pool.row_segments(1)
            pool.prune_slack(slack)
            out = []
            for fused in modes:
                pool.launch_config(fused=fused)
                pool.step(2)
                out.append(np.array(pool.scenario_get(0)))
            return out + [pool.download(s)[0] for s in slots]
    for x, y in zip(run((2, 1, 2, 1)), run((0, 0, 0, 0))):
        assert np.array_equal(x, y)


# a call of no steps leaves the patches' estimates of the step before
@pytest.mark.parametrize("form", ["step", "step_per_patch"])
def test_no_steps_keep_the_estimates(form):
    def run(call):
        pool, slots = _pool(16, 3, 3)
        with pool:
            pool.step(3)
            if call:
                getattr(pool, form)(0)
            return [pool.description(s).estimated_next_timestep_size for s in slots]
    a, b = run(True), run(False)
    assert a == b and min(b) > 0.0

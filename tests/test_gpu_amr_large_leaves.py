"""The batched AMR step and its local time stepping over a hilly bottom with
leaves above 27^2 (more than 8 wavefronts a task from 33 rows on) against the
oracle's AMR driver with the same level-transfer semantics, and a plan of more
tasks than the update reads minima of, against the same calls made one by one
on a flat bottom.  Bitwise: the operations are the same."""
import numpy as np
import pytest

from amr_oracle import OracleBackend
from oracle_lib import wave_propagation_solver

pytestmark = pytest.mark.gpu


def _pair(pool, n):
    from peanoclaw_amd.amr import DeviceBackend, TwoLevelGrid, dam_break_fields
    fn = dam_break_fields(centre=(0.45, 0.52), radius=0.25,
                          hills=[(0.3, 0.6, 0.1, 0.25), (0.7, 0.35, 0.08, 0.2)])
    refined = {(1, 1), (0, 2)}
    dev = TwoLevelGrid(DeviceBackend(pool), 3, 3, n, refined, fn)
    ora = TwoLevelGrid(OracleBackend(), 3, 3, n, refined, fn)
    ora.pure = True
    return dev, ora


def _same(dev, ora):
    a, b = dev.leaf_states(), ora.leaf_states()
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64)), k


@pytest.mark.parametrize("n", [31, 33, 64])
@pytest.mark.parametrize("solver", [1, 2])
def test_global_steps_over_hills(n, solver):
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pool, wave_propagation_solver(solver):
        pool.wave_propagation_solver(solver)
        dev, ora = _pair(pool, n)
        amr = BatchedAmr(dev)
        for _ in range(4):
            assert amr.step(1) == ora.step()
        _same(dev, ora)
        amr.close()


@pytest.mark.parametrize("n", [31, 33, 64])
@pytest.mark.parametrize("solver", [1, 2])
def test_local_time_stepping_over_hills(n, solver):
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pool, wave_propagation_solver(solver):
        pool.wave_propagation_solver(solver)
        dev, ora = _pair(pool, n)
        amr = BatchedAmr(dev)
        amr.lts_init()
        for _ in range(6):
            assert amr.lts_iterations(1, 1.0) == ora.lts_iteration(1.0)
        for p, q in zip(dev.leaves, ora.leaves):
            assert dev.b.clock(p.handle) == ora.b.clock(q.handle)
        _same(dev, ora)
        amr.close()


def test_more_tasks_than_minima_at_once():
    """1097 leaves of 33^2, a task each: their minima are folded first."""
    from peanoclaw_amd.amr import BatchedAmr, DeviceBackend, TwoLevelGrid, dam_break_fields
    from peanoclaw_amd.pool import PatchPool
    fn = dam_break_fields(centre=(0.45, 0.52), radius=0.25)
    with PatchPool(0) as pa, PatchPool(0) as pb:
        one, dev = [TwoLevelGrid(DeviceBackend(p), 33, 33, 33, {(16, 25)}, fn) for p in (pa, pb)]
        amr = BatchedAmr(dev)
        for _ in range(2):
            assert amr.step(1) == one.step()
        for p, q in zip(one.leaves, dev.leaves):
            assert np.array_equal(pa.download(p.handle)[0], pb.download(q.handle)[0]), p.ij
        amr.close()

"""The batched AMR step and its local time stepping against the same calls
made one by one on the device, over leaf sizes around the row segments' and
lane groups' limits.  On a flat bottom the two forms perform the same
operations (h + b - b is h), so everything is compared bitwise: uNew, uOld
with its ghost ring, and the virtual patches' restricted values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grids(n, solver, pool):
    from peanoclaw_amd.amr import DeviceBackend, TwoLevelGrid, dam_break_fields
    pool.wave_propagation_solver(solver)
    fn = dam_break_fields(centre=(0.45, 0.52), radius=0.25)
    refined = {(1, 1), (0, 2)}
    return [TwoLevelGrid(DeviceBackend(pool), 3, 3, n, refined, fn) for _ in range(2)]


def _same(a, b):
    for lev in a.levels:
        for ij, p in a.levels[lev].items():
            q = b.levels[lev][ij]
            x, y = a.b.pool.download(p.handle), b.b.pool.download(q.handle)
            assert np.array_equal(x[0], y[0]), (lev, ij)
            if p.virtual:
                assert np.array_equal(x[1][:, 1:-1, 1:-1], y[1][:, 1:-1, 1:-1]), (lev, ij)
            else:
                assert np.array_equal(x[1], y[1]), (lev, ij)


@pytest.mark.parametrize("n", [3, 5, 16, 31, 33, 64])
@pytest.mark.parametrize("solver", [1, 2])
def test_global_steps(n, solver):
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pa, PatchPool(0) as pb:
        one, _ = _grids(n, solver, pa)
        dev, _ = _grids(n, solver, pb)
        amr = BatchedAmr(dev)
        for _ in range(3):
            assert amr.step(1) == one.step()
        _same(one, dev)
        amr.close()


@pytest.mark.parametrize("n", [3, 16, 33, 64])
@pytest.mark.parametrize("solver", [1, 2])
def test_local_time_stepping(n, solver):
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pa, PatchPool(0) as pb:
        one, _ = _grids(n, solver, pa)
        dev, _ = _grids(n, solver, pb)
        amr = BatchedAmr(dev)
        amr.lts_init()
        for _ in range(6):
            assert amr.lts_iterations(1, 1.0) == one.lts_iteration(1.0)
        for p in dev.leaves:
            q = one.levels[p.level][p.ij]
            assert dev.b.clock(p.handle) == one.b.clock(q.handle)
            assert np.array_equal(dev.b.pool.download(p.handle)[0],
                                  one.b.pool.download(q.handle)[0])
        amr.close()


def test_neighbour_lists_of_any_length():
    """Neighbour lists longer than the usual eight (here every neighbour three
    times) give the same flags."""
    from peanoclaw_amd.amr import BatchedAmr, iarr_list
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pa, PatchPool(0) as pb:
        amrs = []
        for pool in (pa, pb):
            dev, _ = _grids(8, 1, pool)
            amrs.append(BatchedAmr(dev))
            amrs[-1].lts_init()
        g = amrs[1].grid
        ptr, idx = [0], []
        for p in g.leaves:
            idx += [q.handle for q in g._lts[2][p.handle]] * 3
            ptr.append(len(idx))
        assert amrs[1].lib.pc_amr_lts_init(amrs[1].h, iarr_list(ptr), iarr_list(idx)) == 0
        for _ in range(20):
            assert amrs[0].lts_iterations(1, 1.0) == amrs[1].lts_iterations(1, 1.0)
        for p in g.leaves:
            q = amrs[0].grid.levels[p.level][p.ij]
            assert np.array_equal(pb.download(p.handle)[0], pa.download(q.handle)[0])
        for a in amrs:
            a.close()

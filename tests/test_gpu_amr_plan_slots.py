"""A batched AMR plan whose slots change while it lives: a patch of another
size in space (pc_patch_set_description), a slot released and registered again
elsewhere in the pool.  Compared with the same calls made one by one, bitwise:
on a flat bottom the two forms perform the same operations, and doubling every
length is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(pool, n, solver):
    from peanoclaw_amd.amr import DeviceBackend, TwoLevelGrid, dam_break_fields
    from peanoclaw_amd.pool import make_description
    pool.wave_propagation_solver(solver)
    filler = pool.register(make_description((0.0, 0.0), 1.0, 2))
    fn = dam_break_fields(centre=(0.45, 0.52), radius=0.25)
    return filler, TwoLevelGrid(DeviceBackend(pool), 3, 3, n, {(1, 1), (0, 2)}, fn)


def _patches(grid):
    return [p for lev in sorted(grid.levels) for p in grid.levels[lev].values()]


def _double(grid):
    for p in _patches(grid):
        d = grid.b.pool.description(p.handle)
        for k in range(2):
            d.size[k] *= 2.0
            d.position[k] *= 2.0
        grid.b.pool.set_description(p.handle, d)


def _move(grid, filler, p):
    """Patch p's slot registered again on another tile: its old one goes to a
    patch of the same size."""
    pool = grid.b.pool
    d, data, off = pool.description(p.handle), pool.download(p.handle), pool.offset(p.handle)
    pool.release(p.handle)
    pool.release(filler)
    assert pool.register(d) == filler
    assert pool.offset(filler) == off
    assert pool.register(d) == p.handle
    assert pool.offset(p.handle) != off
    pool.upload(p.handle, *data)


def _same(a, b):
    for p, q in zip(_patches(a), _patches(b)):
        x, y = a.b.pool.download(p.handle), b.b.pool.download(q.handle)
        assert np.array_equal(x[0], y[0]), (p.level, p.ij)
        if not p.virtual:
            assert np.array_equal(x[1], y[1]), (p.level, p.ij)


def _run(n, solver, change, lts):
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool
    with PatchPool(0) as pa, PatchPool(0) as pb:
        (fa, one), (fb, dev) = _grid(pa, n, solver), _grid(pb, n, solver)
        amr = BatchedAmr(dev)
        if lts:
            amr.lts_init()
        for k in range(4):
            if k == 2:
                change(one, fa)
                change(dev, fb)
            if lts:
                assert amr.lts_iterations(1, 1.0) == one.lts_iteration(1.0)
            else:
                assert amr.step(1) == one.step()
        if not lts:
            _same(one, dev)
        for p, q in zip(one.leaves, dev.leaves):
            assert np.array_equal(pa.download(p.handle)[0], pb.download(q.handle)[0]), p.ij
        amr.close()


# 33: more than 8 wavefronts a task
@pytest.mark.parametrize("n", [16, 33])
@pytest.mark.parametrize("solver", [1, 2])
@pytest.mark.parametrize("lts", [False, True])
def test_resized(n, solver, lts):
    _run(n, solver, lambda g, filler: _double(g), lts)


@pytest.mark.parametrize("kind", ["coarse leaf", "fine leaf", "virtual"])
@pytest.mark.parametrize("lts", [False, True])
def test_moved(kind, lts):
    def change(g, filler):
        p = {"coarse leaf": g.levels[1][(1, 0)], "fine leaf": g.levels[2][(3, 4)],
             "virtual": g.levels[1][(1, 1)]}[kind]
        _move(g, filler, p)
    _run(16, 1, change, lts)


def test_other_cell_counts_are_refused():
    from peanoclaw_amd.amr import BatchedAmr
    from peanoclaw_amd.pool import PatchPool, make_description
    for at in ((1, 1), (1, 0)):  # a virtual patch, a leaf
        with PatchPool(0) as pool:
            _, g = _grid(pool, 16, 1)
            amr = BatchedAmr(g)
            amr.step(1)
            p = g.levels[1][at]
            d = pool.description(p.handle)
            pool.release(p.handle)
            assert pool.register(make_description(p.pos, p.size, 8, ny=16, level=1,
                                                  is_virtual=bool(d.is_virtual))) == p.handle
            with pytest.raises(Exception, match="AMR plan changed"):
                amr.step(1)
            amr.close()

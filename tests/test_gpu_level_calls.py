"""Batches of interpolations and restrictions against the same calls one by
one: groups of one call, long groups, and calls joined by few links (which
run wave by wave instead of as one group), over patch sizes around the
workgroup's.  Bitwise: a batch is exactly its sequence."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ip(v):
    a = np.ascontiguousarray(np.asarray(v, dtype=np.int32).ravel())
    return a, a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


def _pool(n, parents, children, virtual):
    """Patches of n x n cells: `parents` on the unit square (all at the same
    place) and `children` on its thirds in turn, random data and b."""
    from peanoclaw_amd.pool import PatchPool, make_description
    rng = np.random.default_rng(n)
    pool = PatchPool(0)
    out = []
    for k in range(parents + children):
        c = k - parents
        if c < 0:
            d = make_description((0.0, 0.0), 1.0, n, level=1, time=0.2, timestep_size=0.05,
                                 is_virtual=virtual)
        else:
            d = make_description((c % 3 / 3.0, c // 3 % 3 / 3.0), 1.0 / 3.0, n, level=2,
                                 time=0.21, timestep_size=0.01)
        s = pool.register(d)
        pool.upload(s, unew=rng.uniform(0.5, 2.0, (3, n, n)),
                    uold=rng.uniform(0.5, 2.0, (3, n + 2, n + 2)),
                    b=rng.uniform(0.0, 0.3, (n + 2, n + 2)))
        out.append(s)
    return pool, out[:parents], out[parents:]


def _same(pa, pb, slots):
    for s in slots:
        for x, y in zip(pa.download(s), pb.download(s)):
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), s


def _shapes(k):
    """(source, destination) pairs of a batch over 7 parents and 9 children."""
    if k == "apart":
        return [(i, i) for i in range(7)]
    if k == "one parent":
        return [(0, i) for i in range(9)] * 2
    return [(i, i) for i in range(7)] + [(i + 1, i) for i in range(6)]  # joined, two waves


@pytest.mark.parametrize("n", [6, 23, 33, 64])
@pytest.mark.parametrize("shape", ["apart", "one parent", "joined"])
def test_interpolations(n, shape):
    (pa, P, C), (pb, _, _) = _pool(n, 7, 9, False), _pool(n, 7, 9, False)
    calls = [((n, n), (0, 0), P[s], C[d], k % 2, k % 2, 0)
             for k, (s, d) in enumerate(_shapes(shape))]
    for c in calls:
        assert pa.lib.pc_interpolate_solution(pa.h, (ctypes.c_int * 2)(*c[0]),
                                              (ctypes.c_int * 2)(*c[1]), *c[2:]) == 0
    a = [_ip(v) for v in ([c[0] for c in calls], [c[1] for c in calls], [c[2] for c in calls],
                          [c[3] for c in calls], [c[4:] for c in calls])]
    assert pb.lib.pc_interpolate_batch(pb.h, len(calls), *(p for _, p in a)) == 0
    _same(pa, pb, P + C)


@pytest.mark.parametrize("n", [6, 23, 33, 64])
@pytest.mark.parametrize("shape", ["apart", "one parent", "joined"])
def test_restrictions(n, shape):
    (pa, P, C), (pb, _, _) = _pool(n, 7, 9, True), _pool(n, 7, 9, True)
    pairs = [(C[d], P[s]) for s, d in _shapes(shape)]
    for c, v in pairs:
        assert pa.lib.pc_restrict_solution(pa.h, c, v, 0) == 0
    src, dst = _ip([c for c, _ in pairs]), _ip([v for _, v in pairs])
    assert pb.lib.pc_restrict_batch(pb.h, len(pairs), src[1], dst[1], 0) == 0
    for v in P:
        for pool in (pa, pb):
            assert pool.lib.pc_post_process_restriction(pool.h, v, 0) == 0
    _same(pa, pb, P + C)

"""Batched AMR plans in a pool whose budget leaves no room for the list of the
restriction's contributions (steps derive them) against plans that keep it,
bitwise: state, clocks and the virtual patches."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(px, n, lts, budget):
    from peanoclaw_amd.amr import AmrGrid, BatchedAmr, DeviceBackend, wet_dry_fields
    from peanoclaw_amd.pool import PatchPool, tile_stride
    patches = px * px * (1 + 9 + 81)
    cells = patches * ((n + 2) * tile_stride(n) + 16)
    with PatchPool(0, 56 * cells if budget else 0) as pool:
        pool.reserve(cells)
        # two levels of refinement everywhere: two virtual patches above a leaf
        g = AmrGrid(DeviceBackend(pool), px, px, n, lambda lev, ij: True, wet_dry_fields(),
                    max_level=3)
        free = torch.cuda.mem_get_info()[0]
        amr = BatchedAmr(g)
        taken = free - torch.cuda.mem_get_info()[0]
        if lts:
            amr.lts_init()
            steps = [amr.lts_iterations(1, 1.0) for _ in range(3)]
        else:
            steps = [amr.step(2) for _ in range(2)]
        out = [pool.download(p.handle) for lev in g.levels.values() for p in lev.values()]
        amr.close()
        return steps, out, taken


# 10.6 M contributions of 16 bytes are more than the list every plan may have
@pytest.mark.parametrize("lts", [False, True])
def test_no_room_for_the_list(lts):
    (sa, a, tight), (sb, b, roomy) = _run(4, 64, lts, True), _run(4, 64, lts, False)
    assert tight < 16 * 2 * 16 * 81 * 64 * 64 <= roomy
    assert sa == sb
    for x, y in zip(a, b):
        assert np.array_equal(x[0], y[0])
        assert np.array_equal(x[1], y[1])

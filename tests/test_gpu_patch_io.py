"""pc_patch_upload / pc_patch_download: what goes up comes down, array by
array, for patch sizes at the limits of tiles and workgroups; arrays that are
not given keep their values, and so do the neighbouring tiles."""
import numpy as np
import pytest

from peanoclaw_amd.pool import PatchPool, make_description

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 64), (64, 3), (7, 8), (16, 16), (64, 64)])
def test_round_trip(nx, ny):
    rng = np.random.default_rng(nx * 100 + ny)

    def arrays():
        return [rng.uniform(-1, 1, (3, nx, ny)), rng.uniform(-1, 1, (3, nx + 2, ny + 2)),
                rng.uniform(-1, 1, (nx + 2, ny + 2))]
    with PatchPool(0) as pool:
        slots = [pool.register(make_description((k, 0.0), 1.0, nx, ny=ny)) for k in range(3)]
        held = []
        for s in slots:
            held.append(arrays())
            pool.upload(s, *held[-1])
        for what in range(8):
            new = arrays()
            pool.upload(slots[1], *[a if what >> k & 1 else None for k, a in enumerate(new)])
            held[1] = [a if what >> k & 1 else h for k, (a, h) in enumerate(zip(new, held[1]))]
            for s, h in zip(slots, held):
                for x, y in zip(pool.download(s), h):
                    assert np.array_equal(x, y)

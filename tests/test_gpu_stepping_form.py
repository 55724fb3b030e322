"""Which kernel a 3D domain steps with (Domain.tile): a tile that the caller
sets is the one that runs wherever the results do not depend on it, tuning
keeps whole rows only where they serve, and the separable form is by the grid
alone."""
import numpy as np
import pytest

import test_gpu_separable3d as sep
from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu

STORED = [("f32", False), ("f16", True), ("bf16", False), ("f16u", True)]


def field(n, seed):
    rng = np.random.default_rng(seed)
    return wl.equilibrium_moments(rng.uniform(-0.05, 0.05, (n, 3)), rng.uniform(0.98, 1.02, n)).astype(np.float32)


@pytest.mark.parametrize("storage,fast", STORED)
def test_set_tile_is_the_one_that_runs(storage, fast):
    grid = (190, 121, 65)
    print(f"case set tile {grid} {storage} fast={fast}", flush=True)
    d = [capi.Domain(3, *grid, viscosity=0.02, storage=storage, periodic=True, fast_math=fast) for _ in range(3)]
    for x in d:
        x.set_moments(field(x.n, 5))
    assert d[0].tile()[0] == capi.FORM_ROWS
    d[1].set_tile(9)
    assert d[1].tile() == (capi.FORM_TILES, 9)
    t = d[2].autotune()
    assert d[2].tile() in ((capi.FORM_TILES, t), (capi.FORM_ROWS, t)) and 0 <= t < 16
    for x in d:
        x.step(3)
    want = d[0].moments(0)
    for x in d[1:]:
        assert np.array_equal(x.moments(0), want)
        x.close()
    d[0].close()


def test_tuning_after_a_set_tile_may_take_the_rows_again():
    """256x192x160 in FP16: rows 113 us a step, 147 the best tile, 350 the boxes."""
    d = capi.Domain(3, 256, 192, 160, viscosity=0.02, storage="f16", periodic=True, fast_math=True)
    d.set_moments(field(d.n, 6))
    d.set_tile(0)
    assert d.tile() == (capi.FORM_TILES, 0)
    d.autotune()
    assert d.tile()[0] == capi.FORM_ROWS
    d.close()


def test_separable_form_is_by_the_grid():
    grid = sep.GRIDS[0]
    a, b = (capi.Domain(3, *grid, viscosity=0.02, fast_math=True) for _ in range(2))
    for x in (a, b):
        x.set_moments(field(x.n, 7))
    b.set_tile(9)
    t = b.autotune()
    assert b.tile() == (capi.FORM_SEPARABLE, 9) and t == 9 and a.tile()[0] == capi.FORM_SEPARABLE
    for x in (a, b):
        x.step(3)
    assert np.array_equal(a.moments(0), b.moments(0))
    f = np.ones(grid[::-1], np.uint8)
    f[:, 0, :] = 5  # a bounce-back wall
    b.set_flags(f.ravel())
    assert b.tile() == (capi.FORM_TILES, 9)
    v, e = wl.icosphere([g / 2 for g in grid], 6.3, 1)
    a.set_boundary(v.astype(np.float32), np.zeros_like(v, np.float32), e)
    assert a.tile()[0] == capi.FORM_TILES
    for x in (a, b):
        x.close()

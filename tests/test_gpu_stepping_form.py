"""Which kernel a 3D domain steps with (Domain.tile): a tile that the caller
sets is the one that runs wherever the results do not depend on it, tuning
keeps whole rows only where they serve, and the separable form is by the grid
alone.  The tests of the whole-row kernels reach them on the grids that they
name; the columns keep a full-grid comparison in both arithmetic forms."""
import numpy as np
import pytest

import oracle_lib as ol
import test_gpu_rows3d as rows
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


def test_grids_of_the_whole_row_tests_reach_them():
    for grids, want, kw in ((rows.GRIDS, capi.FORM_ROWS, [dict(storage=s, fast_math=f) for s, f in
                                                          [("f32", False), ("f16", True), ("f16", False), ("bf16", True),
                                                           ("f16u", True), ("f16u", False)]]),
                            (sep.GRIDS + [(127, 50, 90)], capi.FORM_SEPARABLE, [dict(fast_math=True)])):
        for g in grids:
            for k in kw:
                for periodic in (True, False):
                    d = capi.Domain(3, *g, viscosity=0.02, periodic=periodic, **k)
                    assert d.tile()[0] == want, (g, k)
                    d.close()


@pytest.mark.parametrize("grid", [(276, 201, 10), (277, 202, 86)])
@pytest.mark.parametrize("periodic", [True, False])
def test_fast_fp32_rows_equal_columns(grid, periodic):
    """Grids whose rows serve where the separable form does not."""
    print(f"case fast rows {grid} periodic={periodic}", flush=True)
    m, f = rows.setup(grid, 9, periodic)
    d = [capi.Domain(3, *grid, viscosity=0.02, periodic=periodic, fast_math=True) for _ in range(2)]
    for x in d:
        x.set_flags(f)
        x.set_moments(m)
    d[1].set_tile(7)
    assert [x.tile()[0] for x in d] == [capi.FORM_ROWS, capi.FORM_TILES]
    for x in d:
        x.step(5)
    assert np.array_equal(d[0].moments(0), d[1].moments(0))
    for x in d:
        x.close()


def test_columns_on_a_full_grid_with_a_wall():
    """The 64x4 columns in both forms on 256x128x128 with a wall and a block
    of wall cells, against the FP32 oracle; the fast form within the 1e-5
    relative L2 that it is held to elsewhere."""
    c = wl.TG3D
    grid = (c["nx"], c["ny"], c["nz"])
    print(f"case columns {grid} with a wall", flush=True)
    m = np.asarray(wl.taylor_green_ring(*grid, c["amp"], c["ring_r"], c["seed"]), np.float32)
    f = np.ones(grid[::-1], np.uint8)
    f[:, 0, :] = 5
    f[60:64, 50:55, 100:107] = 3
    ol.set_threads(0)
    o = ol.OracleDomain(3, *grid, fp64=False, stage_fp16=False, periodic=True, nu=c["viscosity"])
    o.set_flags(f.ravel())
    o.set_moments(m.astype(np.float64))
    o.step(20)
    ref = o.moments(0)
    for fast in (False, True):
        d = capi.Domain(3, *grid, viscosity=c["viscosity"], periodic=True, fast_math=fast)
        d.set_flags(f.ravel())
        d.set_tile(9)
        assert d.tile() == (capi.FORM_TILES, 9)
        d.set_moments(m)
        d.step(20)
        got = d.moments(0).astype(np.float64)
        d.close()
        if fast:
            assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
        else:
            assert np.array_equal(got, ref)

"""3D domains whose tile was neither set nor tuned take one by their grid:
the results are those of the box tile bit for bit, on either side of each
step of the rule (cells without and with a body, and both moment buffers
against 256 MB), and a tile that the caller sets is the one that runs."""
import numpy as np
import pytest

from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu


def flow(grid, body, tile, **kw):
    nx, ny, nz = grid
    d = capi.Domain(3, nx, ny, nz, viscosity=0.02, **kw)
    f = np.ones((nz, ny, nx), np.uint8)
    f[:, 0, :] = 5
    d.set_flags(f.ravel())
    rng = np.random.default_rng(8)
    d.set_moments(wl.equilibrium_moments(rng.uniform(-0.02, 0.02, (nx * ny * nz, 3))).astype(np.float32))
    if body:
        v, e = wl.icosphere((nx / 2, ny / 2, nz / 2), 11.3, 1)
        vel = np.tile(np.float32([0.02, -0.01, 0.01]), (len(v), 1))
        d.set_boundary(v.astype(np.float32), vel, e)
    if tile is not None:
        d.set_tile(tile)
    d.step(4)
    out = [d.moments(0)] + ([d.body_wrench(), d.step_vertex_forces()] if body else [])
    d.close()
    return out


@pytest.mark.parametrize("grid,body,kw", [
    ((70, 71, 70), True, {}),
    ((71, 71, 70), True, dict(fast_math=True)),
    ((100, 76, 76), False, {}),
    ((100, 77, 76), False, dict(fast_math=True)),
    ((256, 120, 103), False, {}),
    ((256, 120, 105), True, dict(fast_math=True)),
    ((257, 120, 110), False, {}),
    ((288, 148, 152), True, dict(fast_math=True, storage="f16")),
])
def test_default_tile_equals_box(grid, body, kw):
    print(f"case default tile {grid} body={body} {kw}", flush=True)
    a, b = flow(grid, body, None, **kw), flow(grid, body, 0, **kw)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)

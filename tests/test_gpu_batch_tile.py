"""The tile of a batch is searched on the members that step with tiles: with
none there is no search, and one that comes to the tiles later (a wall in its
flags) is searched for then.  The 8x8x4 boxes (index 0, what no search gives)
take about twice as long as the columns on this grid."""
import numpy as np
import pytest

from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu


def test_tile_is_searched_when_a_member_comes_to_the_tiles():
    nx, ny, nz = 256, 128, 128
    print(f"case batch tile {nx}x{ny}x{nz}", flush=True)
    d = capi.Domain(3, nx, ny, nz, viscosity=0.02, fast_math=True)
    d.set_moments(wl.equilibrium_moments(np.zeros((d.n, 3))).astype(np.float32))
    b = capi.Batch(3, fast_math=True)
    b.add(d)
    b.step(2)
    assert b.tile()[0] == 0
    f = np.ones((nz, ny, nx), np.uint8)
    f[:, 0, :] = 5
    d.set_flags(f.ravel())
    b.step(2)
    assert b.tile()[0] > 0
    b.close()
    d.close()

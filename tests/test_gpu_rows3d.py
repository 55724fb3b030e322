"""The whole-row tile of 3D domains without a body: 64 x 6 cells marching
along z in chunks, with the arithmetic of the staged columns, so every
comparison is bit for bit.  Grids of whole tiles, ragged last columns and
rows, a cell more and less than a tile, chunks of one plane to many; periodic
and clamped sides with inlet, outlet and cells that are not updated.  The
reference order is compared with the CPU oracle, the other forms and storages
with the same domain in a batch, whose tiles are the columns."""
import numpy as np
import pytest

import oracle_lib as ol
from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu

GRIDS = [(64, 301, 57), (190, 121, 65), (250, 138, 33), (512, 61, 33), (126, 18, 801)]


def setup(grid, seed, periodic):
    nx, ny, nz = grid
    rng = np.random.default_rng(seed)
    n = nx * ny * nz
    m = wl.equilibrium_moments(rng.uniform(-0.1, 0.1, (n, 3)), rng.uniform(0.98, 1.02, n))
    m[:, 4:] += rng.uniform(-0.3, 0.3, (n, 6)) * (rng.random((n, 1)) < 0.3)  # some negative populations
    f = np.ones((nz, ny, nx), np.uint8)
    if not periodic:
        f[:, :, 0] = 13  # inlet
        f[:, :, -1] = 20  # outlet
        f[nz // 2, ny // 3, nx // 4 : nx // 2] = 2  # not updated
    return m.astype(np.float32), f.ravel()


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("periodic", [True, False])
def test_reference_order_equals_oracle(grid, periodic):
    print(f"case rows {grid} periodic={periodic}", flush=True)
    m, f = setup(grid, 3, periodic)
    g = capi.Domain(3, *grid, viscosity=0.02, periodic=periodic)
    o = ol.OracleDomain(3, *grid, fp64=False, stage_fp16=False, periodic=periodic, nu=0.02)
    for d in (g, o):
        d.set_flags(f)
    g.set_moments(m)
    o.set_moments(m.astype(np.float64))
    for steps in (1, 4):
        g.step(steps)
        o.step(steps)
        assert np.array_equal(g.moments(0).astype(np.float64), o.moments(0))
    g.close()


@pytest.mark.parametrize("storage,fast", [("f16", True), ("f16", False), ("bf16", True), ("f16u", True), ("f16u", False)])
@pytest.mark.parametrize("grid", GRIDS[1:4])
@pytest.mark.parametrize("periodic", [True, False])
def test_equals_columns(storage, fast, grid, periodic):
    print(f"case rows {grid} {storage} fast={fast} periodic={periodic}", flush=True)
    m, f = setup(grid, 4, periodic)
    b = capi.Batch(3, storage, periodic=periodic, fast_math=fast)
    b.set_tile(7)
    d = [capi.Domain(3, *grid, viscosity=0.02, storage=storage, periodic=periodic, fast_math=fast) for _ in range(2)]
    for x in d:
        x.set_flags(f)
        x.set_moments(m)
    b.add(d[1])
    d[0].step(5)
    b.step(5)
    b.sync()
    assert np.array_equal(d[0].moments(0), d[1].moments(0))
    b.close()
    for x in d:
        x.close()

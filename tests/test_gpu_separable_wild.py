"""Infinite, huge and NaN moments in the separable 3D form: the cells around
them agree with the reference-order kernels, non-finite ones included, whichever
moment it is and wherever the cell lies among tiles, chunks and grid edges.

After one step every value is finite or not where it is in the reference order;
rho agrees to 1e-5 of itself and u and Pi, sums over non-negative populations
divided by rho and so at most of order one, to 1e-5 (some 40 FP32 roundings of
6e-8).  Infinities and NaN have left the flow after two more steps, and every
moment agrees to 1e-5 again."""
import numpy as np
import pytest

from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu

GRID = (127, 50, 90)
# corners of the grid, both sides of tile edges (64 x 8) and cells inside
AT = [(0, 0, 0), (126, 49, 89), (63, 7, 20), (64, 16, 31), (20, 15, 40), (100, 24, 53), (0, 31, 60), (126, 8, 70),
      (50, 49, 12), (90, 0, 80)]


def start():
    n = GRID[0] * GRID[1] * GRID[2]
    rng = np.random.default_rng(6)
    m = wl.equilibrium_moments(rng.uniform(-0.05, 0.05, (n, 3)), rng.uniform(0.98, 1.02, n)).astype(np.float32)
    return m.reshape(GRID[::-1] + (10,))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38, 1e20, -50.0])
@pytest.mark.parametrize("first", [0, 3, 7])
@pytest.mark.parametrize("periodic", [True, False])
@np.errstate(invalid="ignore")
def test_agrees_with_the_reference_order(value, first, periodic):
    print(f"case separable wild {value} first={first} periodic={periodic}", flush=True)
    m = start()
    for k, (x, y, z) in enumerate(AT):
        m[z, y, x, (first + k) % 10] = value
    d = [capi.Domain(3, *GRID, viscosity=0.02, periodic=periodic, fast_math=f) for f in (True, False)]
    assert d[0].tile()[0] == capi.FORM_SEPARABLE
    for x in d:
        x.set_moments(m.reshape(-1, 10))
        x.step(1)
    a, b = (x.moments(0).astype(np.float64) for x in d)
    fin = np.isfinite(b)
    assert np.array_equal(np.isfinite(a), fin)
    assert np.abs(a - b)[fin[:, 0], 0].max() <= 1e-5 * np.abs(b[fin[:, 0], 0]).max()
    near = np.abs(b[:, 0]) < 10  # rho of the flow's own order: relative to itself
    assert np.abs(a - b)[near, 0].max() <= 1e-5
    assert np.abs(a - b)[:, 1:][fin[:, 1:]].max() <= 1e-5
    if not np.isfinite(value):
        for x in d:
            x.step(2)
        a, b = (x.moments(0) for x in d)
        assert np.isfinite(b).all() and np.isfinite(a).all()
        assert np.abs(a - b).max() <= 1e-5
    for x in d:
        x.close()

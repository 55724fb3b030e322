"""The axis-by-axis form of the fast 3D step (whole grids of enough cells,
no body, no bounce-back walls).

Its tile is 64 x 8 cells marching along z in chunks: the cases are whole
tiles, ragged last columns and rows, one chunk, chunks of one to three planes
and one-plane remainders, with periodic and clamped sides, inlet, outlet and
cells that are not updated.  Moments stay within 1e-5 relative L2 of the FP32
oracle after 10 steps, the bound that the other fast forms are held to (a step
carries about 40 FP32 roundings of 6e-8 a cell, signs mixed), and their mass within 2e-8 a cell of its start: the form's
rounding has no bias.
"""
import numpy as np
import pytest

import oracle_lib as ol
from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu

GRIDS = [(64, 128, 64), (127, 50, 90), (254, 99, 25), (1024, 26, 16), (1000, 33, 17), (3000, 33, 9)]


def field(grid, seed, u=0.05, pi=0.0):
    rng = np.random.default_rng(seed)
    n = grid[0] * grid[1] * grid[2]
    m = wl.equilibrium_moments(rng.uniform(-u, u, (n, 3)), rng.uniform(0.98, 1.02, n))
    if pi:
        m[:, 4:] += rng.uniform(-pi, pi, (n, 6))
    return m.astype(np.float32)


def pair(grid, m, flags=None, periodic=False):
    nx, ny, nz = grid
    g = capi.Domain(3, nx, ny, nz, viscosity=0.02, periodic=periodic, fast_math=True)
    o = ol.OracleDomain(3, nx, ny, nz, fp64=False, stage_fp16=False, periodic=periodic, nu=0.02)
    for d in (g, o):
        if flags is not None:
            d.set_flags(flags)
    g.set_moments(m)
    o.set_moments(m.astype(np.float64))
    return g, o


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("periodic", [True, False])
def test_matches_oracle(grid, periodic):
    print(f"case separable {grid} periodic={periodic}", flush=True)
    nx, ny, nz = grid
    flags = np.ones((nz, ny, nx), np.uint8)
    if not periodic:
        flags[:, :, 0] = 13  # inlet
        flags[:, :, -1] = 20  # outlet
        flags[nz // 2, ny // 3, nx // 4 : nx // 2] = 2  # not updated
    g, o = pair(grid, field(grid, 3), flags.ravel(), periodic)
    g.step(10)
    o.step(10)
    e = [rel(g.moments(w), o.moments(w)) for w in (0, 1)]
    print(f"  rel L2 {e[0]:.2e}", flush=True)
    assert max(e) <= 1e-5
    if periodic:  # sum of rho is conserved
        n = nx * ny * nz
        m0 = field(grid, 3)[:, 0].astype(np.float64).sum()
        assert abs(g.moments(0)[:, 0].astype(np.float64).sum() - m0) <= 2e-8 * n
    g.close()


@pytest.mark.parametrize("periodic", [True, False])
def test_negative_populations_are_clamped(periodic):
    """A rough state with many negative populations beside a smooth one.  With
    a NaN cell, whose populations the clamp turns into zeros, the form agrees
    with the reference-order kernels."""
    grid = (127, 50, 90)
    nx, ny, nz = grid
    print(f"case separable clamp periodic={periodic}", flush=True)
    m = field(grid, 4, u=0.25, pi=0.4).reshape(nz, ny, nx, 10)
    m[:30] = field(grid, 3).reshape(nz, ny, nx, 10)[:30]
    g, o = pair(grid, m.reshape(-1, 10), periodic=periodic)
    for steps in (1, 2):
        g.step(steps)
        o.step(steps)
        e = rel(g.moments(0), o.moments(0))
        print(f"  rel L2 {e:.2e}", flush=True)
        assert e <= 1e-5
    m[15, 10, 20, 1] = np.nan
    r = capi.Domain(3, nx, ny, nz, viscosity=0.02, periodic=periodic)
    for d in (g, r):
        d.set_moments(m.reshape(-1, 10))
        d.step(2)
    a, b = g.moments(0), r.moments(0)
    assert np.array_equal(np.isfinite(a), np.isfinite(b))
    assert rel(np.nan_to_num(a), np.nan_to_num(b).astype(np.float64)) <= 1e-5
    r.close()
    g.close()


@pytest.mark.parametrize("periodic", [True, False])
def test_batch_member_equals_alone(periodic):
    """Members of both forms in one batch (the second grid is too small for
    the axis-by-axis form), and a flag change that moves one to the tiles."""
    grids = [(127, 50, 90), (40, 30, 20), (254, 99, 25)]
    print(f"case separable batch periodic={periodic}", flush=True)
    b = capi.Batch(3, periodic=periodic, fast_math=True)
    mem, alone = [], []
    for k, s in enumerate(grids):
        for lst in (mem, alone):
            d = capi.Domain(3, *s, viscosity=0.02, periodic=periodic, fast_math=True)
            d.set_moments(field(s, 7 + k))
            lst.append(d)
        b.add(mem[-1])

    def check():
        b.step(7)
        b.sync()
        for k, (d, a) in enumerate(zip(mem, alone)):
            a.step(7)
            assert np.array_equal(d.moments(0), a.moments(0)), f"member {k}"

    check()
    f = np.ones(grids[2][::-1], np.uint8)
    f[:, 0, :] = 5
    for lst in (mem, alone):
        lst[2].set_flags(f.ravel())
    check()
    b.close()
    for d in mem + alone:
        d.close()

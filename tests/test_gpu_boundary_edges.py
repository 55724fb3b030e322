"""Element sums and link detection at the edges of their work split.

2D takes 16 lanes per segment and two window cells per lane and pass (alone:
16 lanes per segment and direction); 3D takes a 256-thread block per triangle,
two window cells per thread and pass in the detection, and LDS lists of 4096
links.  The cases sit on those edges: element counts around a multiple of 16,
windows of less than a lane row up to several passes, and triangles whose
windows overflow the lists.  Moments are compared with the oracle bit for bit;
forces to 1e-5 relative L2, the bound that an FP32 link force summed in FP64
here and in the oracle's order meets by far (each link force carries a few
FP32 roundings, 1e-7 each, and forces on a body moving against the fluid do
not cancel).
"""
import numpy as np
import pytest

import oracle_lib as ol
from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu


def run_pair(dim, grid, v, vel, e, steps, batched, **kw):
    nx, ny, nz = grid
    g = capi.Domain(dim, nx, ny, nz, viscosity=0.02, **kw)
    o = ol.OracleDomain(dim, nx, ny, nz, fp64=False, stage_fp16=dim == 2, nu=0.02, cf=capi.cf_of(dim, 1.0, 1.0, 1.0))
    rng = np.random.default_rng(5)
    m = wl.equilibrium_moments(rng.uniform(-0.01, 0.01, (nx * ny * nz, dim))).astype(np.float32)
    g.set_moments(m)
    o.set_moments(m.astype(np.float64))
    g.set_boundary(v, vel, e)
    o.set_boundary(v, vel, e)
    b = None
    if batched:
        b = capi.Batch(dim)
        b.add(g)
    for _ in range(steps):
        o.zero_vertex_forces()
        o.step(1)
    if batched:
        b.step(steps)
        b.sync()
    else:
        g.step(steps)
    assert np.array_equal(g.moments().astype(np.float64), o.moments())
    f, fo = g.step_vertex_forces().astype(np.float64), o.vertex_forces()
    assert np.linalg.norm(fo) > 0
    assert np.linalg.norm(f - fo) <= 1e-5 * np.linalg.norm(fo)
    w = g.body_wrench()[0]
    assert np.linalg.norm(w[:dim] - fo.sum(0)) <= 1e-5 * np.abs(fo).sum()
    out = (f, w)
    if b is not None:
        b.close()
    g.close()
    return out


@pytest.mark.parametrize("n_seg,r", [(3, 20.0), (7, 21.3), (15, 9.0), (16, 9.0), (17, 9.0), (33, 14.0), (400, 14.0)])
def test_segments_2d(n_seg, r):
    print(f"case 2D polygon {n_seg} r={r}", flush=True)
    v, e = wl.cylinder(n_seg, 31.3, 29.6, r)
    vel = np.tile([0.02, -0.01], (n_seg, 1))
    a = run_pair(2, (64, 60, 1), v, vel, e, 3, False)
    b = run_pair(2, (64, 60, 1), v, vel, e, 3, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("subdiv,r", [(0, 13.0), (0, 2.2), (1, 13.0), (2, 9.0)])
def test_triangles_3d(subdiv, r):
    print(f"case 3D icosphere {subdiv} r={r}", flush=True)
    v, e = wl.icosphere([17.3, 16.2, 15.6], r, subdiv)
    vel = np.tile([0.02, -0.01, 0.015], (len(v), 1))
    a = run_pair(3, (36, 33, 32), v, vel, e, 2, False)
    b = run_pair(3, (36, 33, 32), v, vel, e, 2, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])

"""Element sums and link detection by the fineness of the mesh, against the
oracle (bounds as in test_gpu_boundary_edges), alone and in a batch with the
same bits.  2D: a block per segment where one is long, beside short ones and
across the grid's edge.  3D: a wave per triangle, which meshes of many small
triangles take in place of a block per triangle: element counts that are no
multiple of the four waves of a block, windows of one pass of a wave to many,
lists that overflow, and the same bits as the block form."""
import numpy as np
import pytest

from freeflow_amd import capi, workloads as wl
from test_gpu_boundary_edges import run_pair

pytestmark = pytest.mark.gpu


def bodies(*parts):
    """One mesh of several (vertices, elements); returns it with the body of each element."""
    v = np.concatenate([p[0] for p in parts])
    off = np.cumsum([0] + [len(p[0]) for p in parts])
    e = np.concatenate([p[1] + o for p, o in zip(parts, off)]).astype(np.uint32)
    return v, e, np.repeat(np.arange(len(parts)), [len(p[1]) for p in parts]).astype(np.int32)


@pytest.mark.parametrize("n_seg,r,n_short", [(3, 20.0, 0), (4, 27.3, 0), (5, 44.0, 0), (3, 24.0, 301)])
def test_long_segments(n_seg, r, n_short):
    print(f"case long segments {n_seg} r={r} beside {n_short}", flush=True)
    v, e = wl.cylinder(n_seg, 31.3, 29.6, r)
    if n_short:
        v, e, _ = bodies((v, e), wl.cylinder(n_short, 30.2, 28.9, 11.0))
    vel = np.tile([0.02, -0.01], (len(v), 1))
    a = run_pair(2, (64, 60, 1), v, vel, e, 3, False)
    b = run_pair(2, (64, 60, 1), v, vel, e, 3, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("drop,big", [(0, None), (1, None), (2, None), (3, 13.0), (0, 9.0)])
def test_fine_meshes(drop, big):
    print(f"case fine mesh drop={drop} big={big}", flush=True)
    v, e = wl.icosphere([17.3, 16.2, 15.6], 6.5 if big is None else 3.7, 3)
    e = e[:len(e) - drop]
    if big is not None:  # 20 triangles whose windows hold hundreds to thousands of cells
        v, e, _ = bodies((v, e), wl.icosphere([18.1, 16.4, 15.2], big, 0))
    vel = np.tile([0.02, -0.01, 0.015], (len(v), 1))
    a = run_pair(3, (36, 33, 32), v, vel, e, 2, False)
    b = run_pair(3, (36, 33, 32), v, vel, e, 2, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_wave_and_block_give_the_same_sums():
    """A body of 20 triangles alone (blocks) and beside a fine one far away
    (waves): its first step is the same."""
    grid = (72, 33, 32)
    print(f"case wave against block {grid}", flush=True)
    big, fine = wl.icosphere([17.3, 16.2, 15.6], 8.2, 0), wl.icosphere([55.1, 16.2, 15.4], 4.1, 3)
    m = wl.equilibrium_moments(np.random.default_rng(3).uniform(-0.02, 0.02, (72 * 33 * 32, 3))).astype(np.float32)
    out = []
    for parts in ((big,), (big, fine)):
        d = capi.Domain(3, *grid, viscosity=0.02)
        d.set_moments(m)
        v, e, b = bodies(*parts)
        d.set_boundary(v, np.tile([0.02, -0.01, 0.015], (len(v), 1)), e, b, len(parts))
        d.set_body_ref(np.tile([17.0, 16.0, 15.0], (len(parts), 1)))
        d.step(1)
        out.append((d.body_wrench()[0], d.body_power()[0], d.step_vertex_forces()[:len(big[0])]))
        d.close()
    assert np.abs(out[0][0]).min() > 0
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("dim", [2, 3])
def test_members_of_different_fineness_equal_alone(dim):
    print(f"case batch of coarse and fine meshes {dim}D", flush=True)
    grid = (64, 60, 1) if dim == 2 else (36, 33, 32)
    if dim == 2:
        meshes = [wl.cylinder(n, 31.3, 29.6, r) for n, r in ((3, 20.0), (60, 12.0), (5, 24.0))]
    else:
        meshes = [wl.icosphere([17.3, 16.2, 15.6], r, s) for r, s in ((9.0, 1), (6.5, 3), (4.0, 2))]
    m = wl.equilibrium_moments(np.random.default_rng(4).uniform(-0.02, 0.02, (int(np.prod(grid)), dim))).astype(np.float32)
    b = capi.Batch(dim)
    pairs = []
    for v, e in meshes:
        pair = [capi.Domain(dim, *grid, viscosity=0.02) for _ in range(2)]
        for d in pair:
            d.set_moments(m)
            d.set_boundary(v, np.tile([0.02, -0.01, 0.015][:dim], (len(v), 1)), e)
        b.add(pair[1])
        pairs.append(pair)
    b.step(3)
    b.sync()
    for alone, member in pairs:
        alone.step(3)
        assert np.array_equal(alone.moments(), member.moments())
        assert np.array_equal(alone.body_wrench(), member.body_wrench()) and np.abs(alone.body_wrench()).min() > 0
        assert np.array_equal(alone.body_power(), member.body_power())
    b.close()
    for pair in pairs:
        for d in pair:
            d.close()

"""Readbacks through pinned memory: flow fields in chunks taken by several
lanes, small results gathered by one kernel, histories in a pinned ring.
Fields of less than one chunk, of whole and of partial ones, one lane and all
of them, equal what was written; readings of several threads do not mix; the
history returns the latest records in order across the ring's end, also where
the ring is too large to be pinned, and rings of many domains that come and go
keep apart."""
import threading

import numpy as np
import pytest

from freeflow_amd import capi, workloads as wl

pytestmark = pytest.mark.gpu


def field(n, nm, seed):
    m = np.random.default_rng(seed).random((n, nm), np.float32) * 0.01
    m[:, 0] += 1
    return m


@pytest.mark.parametrize("dim,grid", [
    (2, (3, 3)),          # less than four records
    (2, (167, 131)),      # one chunk of 512 KB, and a cell more than one
    (2, (21877, 1)),
    (3, (61, 47, 39)),    # two lanes
    (2, (997, 701)),      # just above 16 MB: large chunks
    (3, (128, 96, 71)),   # all lanes, a partial last chunk
])
def test_moments_round_trip(dim, grid):
    print(f"case moments {dim}D {grid}", flush=True)
    d = capi.Domain(dim, *grid, viscosity=0.01, stage_fp16=False)
    m = field(d.n, d.nm, 3)
    d.set_moments(m)
    for which in (0, 1):
        assert np.array_equal(d.moments(which), m)
    d.close()


@pytest.mark.parametrize("storage,tol", [("f16", 1e-5), ("bf16", 1e-4), ("f16u", 1e-5)])
def test_moments_storages(storage, tol):
    """Deviations of 0.01 keep 11 (8) significant bits: 5e-6 (4e-5) of them."""
    d = capi.Domain(3, 61, 47, 39, viscosity=0.01, storage=storage)
    m = field(d.n, d.nm, 4)
    d.set_moments(m)
    a = d.moments()
    assert np.abs(a - m).max() <= tol
    d.set_moments(a)  # stored values come back as they are
    assert np.array_equal(d.moments(), a)
    d.close()


def test_threads():
    """Six threads (more than the idle small blocks kept) read their own domains."""
    doms, want = [], []
    for k in range(6):
        d = capi.Domain(2, 400 + k, 300, viscosity=0.01, stage_fp16=False)
        want.append(field(d.n, d.nm, k))
        d.set_moments(want[-1])
        doms.append(d)
    bad = []

    def work(k):
        for _ in range(10):
            if not np.array_equal(doms[k].moments(), want[k]) or not np.isfinite(doms[k].mass()):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    for d in doms:
        d.close()


@pytest.mark.parametrize("cap", [1, 7, 40000])
def test_history(cap):
    """Every step's wrench and power, read one by one, against the ring."""
    print(f"case history {cap}", flush=True)
    sc = wl.batched_scenes(1, 5)[0]
    d = capi.Domain(**sc.domain_args())
    sc.setup(d, history=cap)
    w, p = [], []
    for _ in range(11):
        d.step(1)
        w.append(d.body_wrench())
        p.append(d.body_power())
    for count in (1, 3, 7, 100):
        n = min(count, cap, 11)
        a, b = d.wrench_history(count), d.power_history(count)
        assert a.shape[0] == n and b.shape[0] == n
        assert np.array_equal(a, np.array(w[-n:])) and np.array_equal(b, np.array(p[-n:]))
    d.close()


def test_histories_of_many_domains():
    """Rings of about 2 KB to 62 KB over several shared slabs, some freed and
    taken again: each returns its own domain's wrench."""
    sc = wl.batched_scenes(1, 5, nx_range=(128, 129), ny_range=(64, 65), seg_range=(40, 41))[0]
    doms = []

    def add(cap):
        d = capi.Domain(**sc.domain_args())
        sc.setup(d, history=cap)
        doms.append(d)

    for k in range(24):
        add(60 + 80 * k)
    for k in (3, 4, 5, 11, 19):
        doms[k].close()
    for k in (19, 11, 5, 4, 3):
        del doms[k]
    for k in range(6):
        add(1900 - 300 * k)
    for k, d in enumerate(doms):
        d.step(1 + k % 3)
    for k, d in enumerate(doms):
        assert np.array_equal(d.wrench_history(4)[-1], d.body_wrench())
        assert np.array_equal(d.power_history(4)[-1], d.body_power())
        d.close()

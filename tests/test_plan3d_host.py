"""The rules that choose how a 3D domain without a tile of its own steps, on
grids on both sides of each line, each measured there (the times stand beside
the rules).  plan3d.h is host code; no GPU needed."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

# grid, separable form?, whole rows (FP32)?, default tile without and with a body (FP32)
CASES = [
    ((256, 128, 128), True, True, 15, 15),
    ((160, 96, 96), True, False, 7, 7),
    ((146, 151, 150), True, False, 7, 7),     # 32x12x16 columns a fifth padding
    ((145, 138, 213), True, False, 7, 7),     # beyond the last-level cache
    ((663, 779, 9), True, True, 15, 15),
    ((64, 128, 64), True, False, 0, 7),
    ((203, 101, 97), False, False, 7, 7),     # separable 53, columns 48 us a step
    ((200, 211, 70), False, False, 7, 7),
    ((17, 13, 3500), False, False, 7, 7),     # padding to 64 cells
    ((1000, 1000, 1), False, False, 7, 7),    # few planes
    ((640, 480, 6), False, False, 7, 7),
    ((1769, 1213, 2), False, False, 15, 15),
    ((211, 105, 125), False, True, 7, 7),
    ((640, 300, 12), False, True, 15, 15),
    ((122, 1398, 4), False, True, 7, 7),
    ((692, 233, 3), False, True, 0, 7),
    ((196, 850, 11), False, False, 15, 15),
    ((64, 64, 64), False, False, 0, 0),
    ((96, 64, 64), False, False, 0, 7),
    ((8, 8, 10000), False, False, 0, 0),      # columns mostly padding
    ((8, 100, 1000), False, False, 0, 0),
    ((24, 8, 4000), False, False, 7, 7),
    ((61, 47, 39), False, False, 0, 0),
    ((1, 1, 1), False, False, 0, 0),
    ((1820, 1820, 32), True, True, 15, 15),   # just below 4 GiB a buffer
    ((1835, 1835, 32), False, False, 15, 15),
]


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan3d") / "check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(HERE, "native", "plan3d_check.cpp"),
                        "-o", exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout

    def of(grids, *args):
        text = "".join("%d %d %d\n" % g for g in grids)
        out = subprocess.run([exe, *args], input=text, stdout=subprocess.PIPE, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return of


def test_grids_on_both_sides_of_each_line(plans):
    for (g, sep, rows, tile, tile_body), p in zip(CASES, plans([c[0] for c in CASES])):
        assert (p[0] > 0, p[1] > 0, p[2], p[3]) == (sep, rows, tile, tile_body), (g, p)


def test_chunks_lie_within_the_grid(plans):
    grids = [(nx, ny, nz) for nx in (1, 63, 65, 640) for ny in (1, 7, 130) for nz in (1, 2, 9, 257, 4001)]
    for g, p in zip(grids, plans(grids)):
        assert 0 <= p[0] <= g[2] and 0 <= p[1] <= g[2] and 0 <= p[4] <= g[2], (g, p)


def test_chunks_of_a_batch_by_all_its_members(plans):
    for grids, planes in (([(64, 128, 64)], 4), ([(64, 128, 64)] * 8, 32), ([(64, 128, 64)] * 32, 64), ([], 1),
                          ([(64, 8, 5), (64, 8, 300)], 2)):
        assert plans(grids, "batch") == [(planes,)], grids

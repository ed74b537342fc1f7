"""The hull routine of the tile kernels against the per-point routine, row by
row, in a host build under AddressSanitizer and UBSan
(tests/cpu_emul/hull_rows.cpp): random points with full, coarse and fine cells,
a near-degenerate lattice, points in rows (many collinear with one another),
close pairs, a cluster, general boxes and exact ties (left to the steps).  Both
tile edges."""
import os
import subprocess

import numpy as np
import pytest

from gpudelaunaytriangulation_amd import inputs
from test_exact_mode import lattice
from test_exact_tile import CSRC, ROOT, off_images, run, twins


@pytest.fixture(scope="module", params=[(5, 2048), (4, 1024)], ids=["ts5", "ts4"])
def exe(request, tmp_path_factory):
    ts, pts = request.param
    out = str(tmp_path_factory.mktemp("hull") / "hull_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-ffp-contract=off", f"-DGDT_TILE_SHIFT={ts}",
                    f"-DGDT_WIN_MAXPTS={pts}", f"-I{CSRC}",
                    os.path.join(ROOT, "tests", "cpu_emul", "hull_rows.cpp"), "-o", out], check=True)
    return out


def in_rows():
    xy = inputs.uniform_points(1600, 40.0, 40.0, seed=12)
    xy[:, 1] = np.floor(xy[:, 1]) + 0.5
    xy[::5, 1] += 0.01 * np.arange(320) / 320.0
    return xy


# name: (points, box x11, x12, x21, x22, cell size)
CASES = {
    "uniform": (lambda: inputs.uniform_points(3000, 70.0, 43.0, seed=5), (70.0, 43.0), 1.0),
    "images": (lambda: off_images(1500, 39.0), (39.0, 39.0), 1.0),
    "coarse": (lambda: inputs.uniform_points(2500, 50.0, 50.0, seed=6), (50.0, 50.0), 1.3),
    "fine": (lambda: inputs.uniform_points(1000, 32.0, 32.0, seed=8), (32.0, 32.0), 0.5),
    "near lattice": (lambda: inputs.lattice_points(64, 64, 1e-5, seed=3), inputs.lattice_box(64, 64), 1.0),
    "rows": (in_rows, (40.0, 40.0), 1.0),
    "close": (lambda: np.delete(twins(), np.s_[450:460], 0)[:450], (30.0, 30.0), 1.0),
    "cluster": (lambda: np.concatenate([inputs.uniform_points(900, 40.0, 40.0, seed=9),
                                        20.0 + inputs.uniform_points(400, 4.0, 4.0, seed=10)]),
                (40.0, 40.0), 1.0),
    "ties": (lambda: lattice(32, 32, 1.0)[0], (32.0, 32.0), 1.0),
    "general": (lambda: inputs.general_points(3000, (55.0, 9.0, 0.0, 55.0), seed=1),
                (55.0, 55.0, 9.0, 0.0), 1.0),
    "left-handed": (lambda: inputs.general_points(2000, (10.0, 48.0, 45.0, 12.0), seed=4),
                    (10.0, 12.0, 48.0, 45.0), 1.1),
    "thin": (lambda: inputs.general_points(1800, (200.0, 30.0, 0.0, 9.0), seed=5),
             (200.0, 9.0, 30.0, 0.0), 1.0),
    "general fine": (lambda: inputs.general_points(1200, (36.0, 8.0, -4.0, 33.0), seed=8),
                     (36.0, 33.0, 8.0, -4.0), 0.5),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_hull_rows_equal_per_point_rows(exe, tmp_path, case):
    gen, box, cell = CASES[case]
    xy = gen()
    n, left, differ, err = run(exe, tmp_path, xy, box[0], box[1], cell, *box[2:])
    assert n == len(xy) and differ == 0 and err == 0
    if case in ("uniform", "images", "near lattice", "general", "thin"):
        assert 10 * left < n        # (the rows come from the hull)
    if case == "ties":
        assert left == n

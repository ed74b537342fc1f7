"""The exact mode's tile and wavefront routines against its per-point routine, row by row, in
a host build under AddressSanitizer and UBSan (tests/cpu_emul/tile_rows.cpp):
random points, lattices off by rounding errors (the double-double decisions),
exact lattices (ties, handed on), coarse and fine cells, a cluster that no
window holds, coincident points, a grid too small for windows and coordinates
outside the box.  Both tile edges."""
import os
import subprocess

import numpy as np
import pytest

from gpudelaunaytriangulation_amd import inputs
from test_exact_mode import lattice

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpudelaunaytriangulation_amd", "csrc")


@pytest.fixture(scope="module", params=[(5, 2048), (4, 1024)], ids=["ts5", "ts4"])
def exe(request, tmp_path_factory):
    ts, pts = request.param
    out = str(tmp_path_factory.mktemp("exact_tile") / "exact_tile")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-ffp-contract=off", f"-DGDT_TILE_SHIFT={ts}",
                    f"-DGDT_WIN_MAXPTS={pts}", f"-I{CSRC}",
                    os.path.join(ROOT, "tests", "cpu_emul", "tile_rows.cpp"), "-o", out], check=True)
    return out


def run(exe, tmp_path, xy, lx, ly, cell, *off_diagonal):
    f = str(tmp_path / "p.bin")
    np.ascontiguousarray(xy, dtype=np.float64).tofile(f)
    out = subprocess.run([exe, f, str(len(xy)), repr(lx), repr(ly), repr(cell),
                          *map(repr, off_diagonal)],
                         capture_output=True, text=True, check=True).stdout.split()
    return [int(v) for v in out]


def off_images(n, L):
    """Uniform points, some of them given up to three boxes away."""
    xy = inputs.uniform_points(n, L, L, seed=31)
    k = np.random.default_rng(7).integers(-3, 4, size=xy.shape)
    return np.where(np.arange(n)[:, None] % 3 == 0, xy + k * L, xy)


def twins():
    xy = inputs.uniform_points(900, 30.0, 30.0, seed=17)
    xy[450:460] = xy[:10]
    xy[460:470] = xy[:10] + 1e-9
    return xy


# name: (points, lx, ly, cell size)
CASES = {
    "uniform": (lambda: inputs.uniform_points(3000, 70.0, 43.0, seed=5), 70.0, 43.0, 1.0),
    "images": (lambda: off_images(1500, 39.0), 39.0, 39.0, 1.0),
    "coarse": (lambda: inputs.uniform_points(2500, 50.0, 50.0, seed=6), 50.0, 50.0, 1.3),
    "fine": (lambda: inputs.uniform_points(1000, 32.0, 32.0, seed=8), 32.0, 32.0, 0.5),
    "decimal": (lambda: lattice(40, 40, 0.1)[0], 4.0, 4.0, 0.1),
    "jitter": (lambda: lattice(36, 36, 0.7)[0] +
               1e-13 * np.random.default_rng(3).standard_normal((36 * 36, 2)), 25.2, 25.2, 0.7),
    "dyadic": (lambda: lattice(32, 32, 1.0)[0], 32.0, 32.0, 1.0),
    "ulps": (lambda: lattice(32, 32, 1.0, 3, 1)[0], 32.0, 32.0, 1.0),
    "cluster": (lambda: np.concatenate([inputs.uniform_points(900, 40.0, 40.0, seed=9),
                                        20.0 + inputs.uniform_points(2100, 2.0, 2.0, seed=10)]),
                40.0, 40.0, 1.0),
    "twins": (lambda: twins()[:460], 30.0, 30.0, 1.5),
    "close": (lambda: np.delete(twins(), np.s_[450:460], 0), 30.0, 30.0, 1.0),
    "tiny": (lambda: inputs.uniform_points(40, 6.0, 6.0, seed=9), 6.0, 6.0, 1.0),
    "tiny60": (lambda: inputs.uniform_points(60, 8.0, 8.0, seed=9), 8.0, 8.0, 1.0),
    "small110": (lambda: inputs.uniform_points(110, 11.0, 11.0, seed=4), 11.0, 11.0, 1.0),
    "far": (lambda: inputs.uniform_points(600, 25.0, 25.0, seed=2) +
            np.where(np.arange(600)[:, None] == 5, 130.0, 0.0), 25.0, 25.0, 1.0),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_tile_rows_equal_per_point_rows(exe, tmp_path, case):
    gen, lx, ly, cell = CASES[case]
    xy = gen()
    n, handed, differ, err = run(exe, tmp_path, xy, lx, ly, cell)
    assert n == len(xy) and differ == 0
    if case in ("uniform", "images", "fine", "jitter"):
        assert 2 * handed < n       # (most rows come from the tile routine)
    if case in ("dyadic", "decimal"):
        assert handed == n          # every point has an exact tie (rectangles)
    if case == "far":
        assert err                  # (every row's flags are compared above)

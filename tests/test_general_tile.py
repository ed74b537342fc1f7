"""The tile routine in general boxes against the per-point routine, row by row,
in a host build under AddressSanitizer and UBSan (tests/cpu_emul/tile_rows.cpp):
mild and strong shear, several periods of it, a rotated and a left-handed
basis, thin boxes, coarse and fine cells, points outside the unit cell, an
exact lattice (ties, handed on), a cluster that no window holds, and a
rectangle.  Both tile edges."""
import numpy as np
import pytest

from gpudelaunaytriangulation_amd import inputs
from test_exact_mode import lattice
from test_exact_tile import exe, run  # noqa: F401  (the fixture)


def pts(n, box, seed):
    return inputs.general_points(n, box, seed=seed)


def outside(box):
    xy = pts(1500, box, 41)
    k = np.random.default_rng(5).integers(-2, 3, size=xy.shape)
    return xy + k @ np.asarray(box).reshape(2, 2).T


def clump(box):
    return np.concatenate([pts(1200, box, 42), 12.0 + inputs.uniform_points(2100, 2.0, 2.0, seed=43)])


C, S = float(np.cos(0.6)), float(np.sin(0.6))
# name: (box x11, x12, x21, x22; points; cell size)
CASES = {
    "mild": ((55.0, 9.0, 0.0, 55.0), lambda b: pts(3000, b, 1), 1.0),
    "strong": ((40.0, -170.0, 0.0, 60.0), lambda b: pts(2400, b, 2), 1.0),
    "rotated": ((45.0 * C, -50.0 * S, 45.0 * S, 50.0 * C), lambda b: pts(2250, b, 3), 1.0),
    "left": ((10.0, 48.0, 45.0, 12.0), lambda b: pts(2000, b, 4), 1.1),
    "thin": ((200.0, 30.0, 0.0, 9.0), lambda b: pts(1800, b, 5), 1.0),
    "hexagonal": ((48.0, 24.0, 0.0, 41.569), lambda b: pts(2000, b, 6), 1.0),
    "coarse": ((44.0, 11.0, 3.0, 42.0), lambda b: pts(1200, b, 7), 1.25),
    "fine": ((36.0, 8.0, -4.0, 33.0), lambda b: pts(1200, b, 8), 0.5),
    "outside": ((40.0, 13.0, 2.0, 39.0), outside, 1.0),
    "clump": ((36.0, 10.0, 0.0, 34.0), clump, 1.0),
    "ties": ((32.0, 64.0, 0.0, 32.0), lambda b: lattice(32, 32, 1.0)[0], 1.0),
    "small": ((16.0, 3.0, 0.0, 15.0), lambda b: pts(240, b, 9), 1.0),
    "rectangle": ((50.0, 0.0, 0.0, 44.0), lambda b: pts(2200, b, 10), 1.0),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_tile_rows_equal_per_point_rows(exe, tmp_path, case):  # noqa: F811
    box, gen, cell = CASES[case]
    xy = gen(box)
    n, handed, differ, err = run(exe, tmp_path, xy, box[0], box[3], cell, box[1], box[2])
    assert n == len(xy) and differ == 0 and err == 0
    if case in ("mild", "strong", "rotated", "hexagonal", "outside"):
        assert 10 * handed < n      # (the rows come from the tile routine)
    if case == "ties":
        assert handed == n

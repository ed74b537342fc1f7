"""The exact mode's star kernel where points tie: a point with two nearest
neighbours is handed on at once, and with it the wave's other points, a block's
together and beyond 256 one by one.  Rows byte for byte those of the per-point
kernel: exact lattices (more points to a block than are kept), a lattice next to
random points, points in pairs of equal distances among random ones, and full
cells, which are handed on too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gpudelaunaytriangulation_amd import inputs  # noqa: E402
from test_exact_mode import lattice  # noqa: E402
from test_gpu_exact_tile import rows  # noqa: E402


def half_lattice():
    xy = lattice(60, 60, 1.0)[0]
    rnd = inputs.uniform_points(3600, 60.0, 60.0, seed=3)
    return np.concatenate([xy[xy[:, 0] < 30.0], rnd[rnd[:, 0] >= 30.0]])


def crosses():
    """Random points, some with four others at one distance (dyadic offsets)."""
    xy = np.floor(inputs.uniform_points(900, 40.0, 40.0, seed=4) * 1024.0) / 1024.0
    d = np.array([[0.125, 0.0], [0.0, 0.125], [-0.125, 0.0], [0.0, -0.125]])
    arms = (xy[:60, None, :] + d[None]).reshape(-1, 2)
    return np.mod(np.concatenate([xy, arms]), 40.0)


def full_cells():
    return np.concatenate([inputs.uniform_points(1200, 40.0, 40.0, seed=5),
                           10.0 + inputs.uniform_points(900, 9.0, 9.0, seed=6)])


# name: (points, side, tile shifts)
CASES = {
    "lattice": (lambda: lattice(64, 64, 1.0)[0], 64.0, (4, 5)),
    "lattice600": (lambda: lattice(600, 600, 1.0)[0], 600.0, (5,)),
    "decimal": (lambda: lattice(72, 72, 0.1)[0] * 10.0, 72.0, (4, 5)),
    "half": (half_lattice, 60.0, (4, 5)),
    "crosses": (crosses, 40.0, (4, 5)),
    "full cells": (full_cells, 40.0, (4, 5)),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_star_rows(case):
    gen, L, shifts = CASES[case]
    xy = gen()
    print(f"[star ties] {case}: n {len(xy)}", flush=True)
    want, wn, _ = rows(xy, L, L, 1.0, tiled=0)
    for ts in shifts:
        got, gn, st = rows(xy, L, L, 1.0, lanes=64, tile_shift=ts)
        assert st["lanes"] == 64
        assert np.array_equal(wn, gn) and np.array_equal(want, got), ts
        if case in ("lattice", "lattice600"):
            assert st["deferred"] == len(xy)
        if case in ("half", "crosses"):
            assert 0 < st["deferred"] < len(xy)

"""An exact tie that a search of the tile routines meets only in the rest of a
circle's cell box, outside its first block of cells: the point is handed on,
as for a tie inside the block.  (The tie's mark taken for an entry would read
the window's arrays before their start, which the sanitizer build reports.)
Lattices in cells a little finer than their spacing, host builds of both tile
edges; the GPU's exact mode against its per-point kernel on the same lattices
and on a triangular one off by rounding errors."""
import numpy as np
import pytest

from test_exact_mode import lattice
from test_exact_tile import exe, run        # noqa: F401  (exe: a fixture)
from test_hull import exe as hull_exe       # noqa: F401

ROW3 = 3.0 ** 0.5 / 2.0


def triangular(nx, ny, jitter=0.0, seed=1):
    col, row = np.meshgrid(np.arange(nx), np.arange(ny), indexing="xy")
    xy = np.stack([col + 0.5 * (row % 2), row * ROW3], -1).reshape(-1, 2)
    xy = xy + jitter * np.random.default_rng(seed).standard_normal(xy.shape)
    return np.mod(xy, [nx, ny * ROW3]), float(nx), ny * ROW3


EXACT = {"square": (lambda: lattice(40, 40, 0.1), 0.09),
         "triangular": (lambda: triangular(24, 24), 0.7),
         "triangular, ulps": (lambda: triangular(24, 24, 1e-15), 0.55)}


@pytest.mark.parametrize("case", sorted(EXACT))
def test_exact_rows(exe, tmp_path, case):       # noqa: F811
    gen, cell = EXACT[case]
    xy, lx, ly = gen()
    n, _, differ, err = run(exe, tmp_path, xy, lx, ly, cell)
    assert n == len(xy) and differ == 0 and err == 0


# (FP64 rows of such a lattice are decided by rounding: only the reads are checked)
@pytest.mark.parametrize("cell", [0.7, 0.55, 0.4])
def test_fp64_steps_stay_in_the_window(hull_exe, tmp_path, cell):       # noqa: F811
    xy, lx, ly = lattice(24, 24, 1.0)
    assert run(hull_exe, tmp_path, xy, lx, ly, cell)[0] == len(xy)


@pytest.mark.parametrize("cell", [0.375, 0.25])
def test_general_steps_stay_in_the_window(exe, tmp_path, cell):         # noqa: F811
    xy, lx, ly = lattice(24, 24, 1.0)
    assert run(exe, tmp_path, xy, lx, ly, cell, 6.0, 0.0)[0] == len(xy)


GPU = dict(EXACT, big=(lambda: triangular(512, 512, 1e-13, 3), 1.0))


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(GPU))
def test_exact_rows_on_the_gpu(case):
    from test_gpu_exact_tile import rows
    gen, cell = GPU[case]
    xy, lx, ly = gen()
    print(f"[tie outside block] {case}: n {len(xy)}", flush=True)
    want, wn, _ = rows(xy, lx, ly, cell, tiled=0)
    for config in ({}, {"lanes": 1, "tile_shift": 5}, {"lanes": 2, "tile_shift": 4},
                   {"lanes": 64, "tile_shift": 4}):
        if config.get("lanes") == 64 and len(xy) > 60000:
            continue
        got, gn, _ = rows(xy, lx, ly, cell, **config)
        assert np.array_equal(wn, gn) and np.array_equal(want, got), config

"""The exact mode's bounds at the ends of the coordinates it takes: neighbours
given as images at opposite ends of the eight box lengths (-4 to +4), on lattices
off by rounding errors.  Every decision taken from an FP64 or double-double value
agrees with the exact sign (the audit build of the host routine); the tile and
wavefront routines' rows are the per-point routine's (host builds under
AddressSanitizer and UBSan), and on the GPU the tile and star kernels' too."""
import numpy as np
import pytest

from test_exact_mode import build_exact_audit, lattice, run_exact_audit
from test_exact_tile import exe, run        # noqa: F401  (exe: a fixture)


def extremes(nx, ny, h, seed, both):
    """A lattice whose points alternate between the images at -4 and +3 box
    lengths in x (both: and in y, by rows)."""
    xy, lx, ly = lattice(nx, ny, h)
    col, row = np.arange(nx * ny) % nx, np.arange(nx * ny) // nx
    kx = np.where((col + row) % 2 == 0, -4.0, 3.0)
    ky = np.where(row % 2 == 0, -4.0, 3.0) if both else np.zeros(nx * ny)
    r = np.random.default_rng(seed)
    kx, ky = [np.where(r.random(nx * ny) < 0.1, r.integers(-4, 4, nx * ny), k) for k in (kx, ky)]
    return xy + np.stack([kx * lx, ky * ly], 1), lx, ly


CASES = {"0.1": (lambda: extremes(16, 16, 0.1, 1, False), 0.1),
         "0.7": (lambda: extremes(18, 14, 0.7, 2, True), 0.7),
         "1.1": (lambda: extremes(15, 15, 1.1, 3, True), 1.1),
         "1": (lambda: extremes(16, 16, 1.0, 4, True), 1.0)}


@pytest.fixture(scope="module")
def audit(tmp_path_factory):
    return build_exact_audit(str(tmp_path_factory.mktemp("audit") / "audit"))


@pytest.mark.parametrize("case", sorted(CASES))
def test_decisions_audited(audit, tmp_path, case):
    (xy, lx, ly), cell = CASES[case][0](), CASES[case][1]
    assert np.abs(xy[:, 0]).max() > 3.9 * lx and (np.abs(xy) <= 4.0 * np.array([lx, ly])).all()
    st, taken, wrong = run_exact_audit(audit, xy, lx, ly, cell, tmp_path)
    assert st == 0 and min(taken) > 0 and wrong == [0, 0, 0]


@pytest.mark.parametrize("case", sorted(CASES))
def test_tile_rows(exe, tmp_path, case):        # noqa: F811
    (xy, lx, ly), cell = CASES[case][0](), CASES[case][1]
    n, _, differ, err = run(exe, tmp_path, xy, lx, ly, cell)
    assert n == len(xy) and differ == 0 and err == 0


@pytest.mark.gpu
@pytest.mark.parametrize("h", [0.1, 0.7, 1.0])
def test_gpu_rows(h):
    from test_gpu_exact_tile import rows
    xy, lx, ly = extremes(60, 56, h, 5, True)
    print(f"[exact extremes] {h}: n {len(xy)}", flush=True)
    want, wn, _ = rows(xy, lx, ly, h, tiled=0)
    for config in ({}, {"lanes": 1, "tile_shift": 5}, {"lanes": 2, "tile_shift": 4}):
        got, gn, _ = rows(xy, lx, ly, h, **config)
        assert np.array_equal(wn, gn) and np.array_equal(want, got), config

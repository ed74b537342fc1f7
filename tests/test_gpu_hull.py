"""The hull kernel (FP64, one lane per point) on the GPU: rows byte for byte
those of the row-major per-point kernel for a global triangulation, and of the
step kernel for a test-and-repair, over both tile edges, block sizes from one wave to sixteen,
sets of a few points to a tile, cells from a quarter of a point to two points
each (with windows that overflow), a near-degenerate lattice, a cluster, exact
ties and a general box."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_FP32F, PREC_FP64, inputs  # noqa: E402
from gpudelaunaytriangulation_amd.delaunay import DelaunayGPU, PeriodicBoundaries  # noqa: E402
from test_exact_mode import lattice  # noqa: E402
from test_gpu_general_tile import cuda, same  # noqa: E402


def rows(xy, moved, box, cell, precision=PREC_FP64, **config):
    """Rows of xy, then of `moved` repaired from them, the number repaired and the statistics."""
    n = len(xy)
    dg = DelaunayGPU(n, 20, cell, PeriodicBoundaries(*box))
    dg.setPrecision(precision)
    dg.ctx.set_config(**config)
    tri = torch.full((n * dg.MaxSize,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(n, dtype=torch.int32, device="cuda")
    dg.globalDelaunayTriangulation(cuda(xy), tri, num)
    st = dg.stats()
    first = tri.cpu().numpy().reshape(n, -1).copy(), num.cpu().numpy().copy()
    dg.testAndRepairDelaunayTriangulation(cuda(moved), tri, num)
    return first, (tri.cpu().numpy().reshape(n, -1), num.cpu().numpy()), dg.last_repaired, st


def square(n, seed):
    L = float(np.sqrt(n))
    return inputs.uniform_points(n, L, L, seed=seed), (L, 0.0, 0.0, L)


def cluster():
    xy, box = square(9000, 6)
    return np.concatenate([xy, 40.0 + inputs.uniform_points(2500, 3.0, 3.0, seed=7)]), box


def near():
    lx, ly = inputs.lattice_box(120, 120)
    return inputs.lattice_points(120, 120, 1e-5, seed=3), (lx, 0.0, 0.0, ly)


BOX = (120.0, 37.0, 0.0, 100.0)
# name: (points and box, cell size)
CASES = {
    "uniform": (lambda: square(30011, 1), 1.0),
    "few": (lambda: square(130, 2), 1.0),
    "fine": (lambda: square(5003, 3), 0.5),
    "full cells": (lambda: square(20021, 4), 1.2),
    "overflow": (lambda: square(20021, 5), 1.45),
    "cluster": (cluster, 1.0),
    "near lattice": (near, 1.0),
    "general": (lambda: (inputs.general_points(12007, BOX, seed=8), BOX), 1.0),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_hull_kernel_rows_equal_per_point_rows(case):
    make, cell = CASES[case]
    xy, box = make()
    print(f"[hull] {case}: n {len(xy)}", flush=True)
    moved = inputs.wrap_into_general_box(
        xy + 0.02 * inputs.gaussian(4, 2 * len(xy)).reshape(-1, 2), box)
    first = rows(xy, xy, box, cell, tiled=0)[0]
    assert int(first[1].sum()) == 6 * len(xy)
    # (what a tile's test flags beside an intruder depends on its windows)
    steps = {ts: rows(xy, moved, box, cell, lanes=2, tile_shift=ts, repair_lanes=2) for ts in (4, 5)}
    for ts, block in ((5, 512), (5, 64), (4, 256), (4, 1024)):
        f, r, c, st = rows(xy, moved, box, cell, lanes=1, tile_shift=ts, repair_lanes=1, block=block)
        assert st["lanes"] == 1
        assert same(first, f) and same(steps[ts][1], r) and c == steps[ts][2], (ts, block)


def test_hull_kernel_ties_take_the_steps():
    xy, lx, ly = lattice(64, 64, 1.0)[:3]
    box = (lx, 0.0, 0.0, ly)
    want, want2, _, _ = rows(xy, xy, box, 1.0, lanes=2, tile_shift=5)
    assert int(want[1].sum()) == 6 * len(xy)
    for ts in (4, 5):
        print(f"[hull] ties, tile shift {ts}", flush=True)
        got, got2, _, _ = rows(xy, xy, box, 1.0, lanes=1, tile_shift=ts, repair_lanes=1)
        assert same(want, got) and same(want2, got2)


@pytest.mark.parametrize("cell", [1.0, 1.2])
def test_filtered_precision_takes_the_hull(cell):
    xy, box = square(30011, 1)
    print(f"[hull] FP32-filtered, cell {cell}", flush=True)
    want, want2, count, _ = rows(xy, xy + 0.01, box, cell, lanes=1, tile_shift=5, repair_lanes=1)
    got, got2, c, _ = rows(xy, xy + 0.01, box, cell, precision=PREC_FP32F, lanes=1, tile_shift=5,
                           repair_lanes=1)
    assert same(want, got) and same(want2, got2) and c == count

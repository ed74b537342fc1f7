"""General boxes through the LDS tile kernels on the GPU: rows byte for byte
those of the row-major per-point kernel, for a global triangulation and a
test-and-repair, over every kernel the dispatch picks (the star kernel, two
lanes and one lane per point, both tile edges), a grid too small for the
windows, a thin box, exact ties, a cluster, and a batch of general and
rectangular boxes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_EXACT, PREC_FP32F, _lib, inputs  # noqa: E402
from gpudelaunaytriangulation_amd.delaunay import (BatchedDelaunayGPU, DelaunayGPU,  # noqa: E402
                                                   PeriodicBoundaries)
from test_exact_mode import lattice  # noqa: E402


def cuda(xy):
    return torch.from_numpy(np.ascontiguousarray(xy)).cuda()


def rows(xy, moved, box, cell, **config):
    """Rows of xy, then of `moved` repaired from them, and the statistics."""
    n = len(xy)
    dg = DelaunayGPU(n, 20, cell, PeriodicBoundaries(*box))
    dg.ctx.set_config(**config)
    tri = torch.full((n * dg.MaxSize,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(n, dtype=torch.int32, device="cuda")
    dg.globalDelaunayTriangulation(cuda(xy), tri, num)
    st = dg.stats()
    first = tri.cpu().numpy().reshape(n, -1).copy(), num.cpu().numpy().copy()
    dg.testAndRepairDelaunayTriangulation(cuda(moved), tri, num)
    return first, (tri.cpu().numpy().reshape(n, -1), num.cpu().numpy()), dg.last_repaired, st


def same(a, b):
    if not np.array_equal(a[1], b[1]):
        return False
    m = np.arange(a[0].shape[1])[None, :] < a[1][:, None]
    return np.array_equal(a[0][m], b[0][m])


# name: (box x11, x12, x21, x22; points; cell size; lanes the automatic choice takes)
CASES = {
    "star": ((65.0, 20.0, 0.0, 63.0), 4100, 1.0, 64),
    "two": ((230.0, -70.0, 10.0, 220.0), 51003, 1.0, 2),
    "one": ((550.0, 171.0, 0.0, 545.0), 300007, 1.0, 1),
    "left": ((30.0, 148.0, 145.0, 12.0), 20011, 1.1, None),
    "sheared": ((100.0, 433.0, 0.0, 90.0), 9001, 1.0, None),
    "thin": ((700.0, 90.0, 0.0, 9.0), 6300, 1.0, None),
    "small": ((6.0, 1.0, 0.0, 6.0), 80, 1.0, None),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_general_tile_rows_equal_per_point_rows(case):
    box, n, cell, lanes = CASES[case]
    print(f"[general tile] {case}: n {n}", flush=True)
    xy = inputs.general_points(n, box, seed=3)
    moved = inputs.wrap_into_general_box(xy + 0.02 * inputs.gaussian(4, 2 * n).reshape(n, 2), box)
    first, repaired, count, _ = rows(xy, moved, box, cell, tiled=0)
    assert int(first[1].sum()) == 6 * n
    configs = [{}, {"lanes": 1, "tile_shift": 5, "repair_lanes": 1}, {"lanes": 4, "tile_shift": 4},
               {"tiled": 2}]
    for config in configs + ([{"lanes": 64, "tile_shift": 5}] if n < 60000 else []):
        f, r, c, st = rows(xy, moved, box, cell, **config)
        if not config and lanes is not None:
            assert st["lanes"] == lanes
        assert same(first, f) and same(repaired, r) and c == count, config


def test_general_tile_ties_and_cluster():
    box = (64.0, 16.0, 0.0, 64.0)
    tie = lattice(64, 64, 1.0)[0]
    clump = np.concatenate([inputs.general_points(4000, box, seed=8),
                            20.0 + inputs.uniform_points(2500, 2.0, 2.0, seed=9)])
    # (sheared by two periods: a square torus, on which ties are exact in FP64)
    for name, xy, b in (("ties", tie, (64.0, 128.0, 0.0, 64.0)), ("cluster", clump, box)):
        print(f"[general tile] {name}", flush=True)
        want, want2, _, _ = rows(xy, xy, b, 1.0, tiled=0)
        assert int(want[1].sum()) == 6 * len(xy)
        got, got2, _, _ = rows(xy, xy, b, 1.0)
        assert same(want, got) and same(want2, got2)


def test_general_tile_mixed_batch():
    boxes = [(50.0, 12.0, 0.0, 48.0), (40.0, 0.0, 0.0, 40.0), (30.0, -9.0, 7.0, 36.0)]
    sizes = [2400, 1600, 1100]
    pts = [inputs.general_points(s, b, seed=50 + i) for i, (s, b) in enumerate(zip(sizes, boxes))]
    print("[general tile] mixed batch", flush=True)
    bd = BatchedDelaunayGPU(sizes, boxes, 20, 1.0, precision=PREC_FP32F)
    tri = torch.full((bd.N * bd.MaxSize,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(bd.N, dtype=torch.int32, device="cuda")
    bd.globalDelaunayTriangulation(cuda(np.concatenate(pts)), tri, num)
    nb, a = tri.cpu().numpy().reshape(bd.N, -1), 0
    for s, b, xy in zip(sizes, boxes, pts):
        want, _, _, _ = rows(xy, xy, b, 1.0, tiled=0)
        mine = nb[a:a + s].copy()
        mine[mine >= 0] -= a
        assert same(want, (mine, num.cpu().numpy()[a:a + s]))
        a += s
    bd.setPrecision(PREC_EXACT)
    with pytest.raises(_lib.GdtError) as e:
        bd.globalDelaunayTriangulation(cuda(np.concatenate(pts)), tri, num)
    assert e.value.status == _lib.GDT_ERR_INVALID

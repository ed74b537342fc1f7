"""Tiles with more points of open triangles than the hull kernel keeps records
for (256; 640 with windows of 4,096 points): cells of 0.5, 0.64, 1.2 and 1.44 points,
and of 2.25, where open points take the steps.  Rows equal to the row-major
per-point kernel's, a global triangulation and a repair of all points, rectangles
and a sheared box; and points on decimal sites, many of them cocircular as far as FP64
tells, where the routine that a point takes can show in its row: it does not
depend on the order of the waves, so every call gives the same rows."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_FP64, _lib, inputs  # noqa: E402
from gpudelaunaytriangulation_amd.delaunay import DelaunayGPU, PeriodicBoundaries  # noqa: E402
from test_gpu_general_tile import cuda, same  # noqa: E402

SLOTS = 24


def triangulate(pts, box, cell, **config):
    n = int(pts.shape[0])
    rect = box[1] == 0.0 and box[2] == 0.0
    dg = DelaunayGPU(n, SLOTS, cell, PeriodicBoundaries(box[0], box[3]) if rect
                     else PeriodicBoundaries(*box))
    dg.ctx.set_config(**config)
    tri = torch.full((n * SLOTS,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(n, dtype=torch.int32, device="cuda")
    dg.globalDelaunayTriangulation(pts, tri, num)
    return dg, tri, num


def host(tri, num):
    return tri.cpu().numpy().reshape(-1, SLOTS).copy(), num.cpu().numpy().copy()


@pytest.mark.parametrize("shear", [0.0, 31.0])
@pytest.mark.parametrize("cell", [0.7, 0.8, 1.1, 1.2, 1.5])
def test_rows_beyond_the_records(cell, shear):
    n, L = 40000, 200.0
    box = (L, shear, 0.0, L)
    pts = cuda(inputs.general_points(n, box, seed=int(10 * cell)))
    print(f"[hull records] cell {cell} shear {shear}", flush=True)
    want = host(*triangulate(pts, box, cell, tiled=0)[1:])
    dg, tri, num = triangulate(pts, box, cell, lanes=1, repair_lanes=1, tile_shift=5)
    assert dg.stats()["lanes"] == 1 and dg.stats()["tile_shift"] == 5
    assert same(want, host(tri, num))
    # every point flagged: the repair rebuilds all rows on the same cell list
    tri.fill_(-7)
    num.zero_()
    flags = torch.zeros(n, dtype=torch.int32, device="cuda")
    req = ctypes.c_int(0)
    st = _lib.load().gdt_repair(dg.ctx.handle, pts.data_ptr(), n, flags.data_ptr(), SLOTS,
                                tri.data_ptr(), num.data_ptr(), PREC_FP64, ctypes.byref(req), None)
    torch.cuda.synchronize()
    assert st == _lib.GDT_OK and same(want, host(tri, num))


@pytest.mark.parametrize("sites,cell", [(10, 0.75), (10, 1.1), (5, 0.7), (5, 1.15), (5, 1.2)])
def test_every_call_gives_the_same_rows(sites, cell):
    """n points on random sites of a grid of spacing 1 / sites."""
    L = 200
    s = np.random.default_rng(5).choice((L * sites) ** 2, L * L, replace=False)
    pts = cuda(np.stack([(s % (L * sites) + 0.5) / sites, (s // (L * sites) + 0.5) / sites], 1))
    print(f"[hull records] sites {sites} cell {cell}", flush=True)
    box = (float(L), 0.0, 0.0, float(L))
    rows = [host(*triangulate(pts, box, cell, lanes=1, tile_shift=5)[1:]) for _ in range(10)]
    assert all(same(rows[0], r) for r in rows[1:])

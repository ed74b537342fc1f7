"""A repair with four lanes per point around the count of flagged points from
which a tile takes two (a quarter of its block's lanes, 64): 0, 1, 63, 64, 65 and all
points of every 16x16-cell tile flagged; rows equal to the triangulation's."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_FP64, _lib, inputs  # noqa: E402
from test_gpu_hull_records import SLOTS, cuda, host, same, triangulate  # noqa: E402


@pytest.mark.parametrize("each", [0, 1, 63, 64, 65, 4096])
@pytest.mark.parametrize("block", [256, 128])
def test_flagged_points_of_a_tile(each, block):
    L, n = 64.0, 4096
    xy = inputs.uniform_points(n, L, L, seed=8)
    tile = (xy[:, 0] // 16).astype(int) + 4 * (xy[:, 1] // 16).astype(int)
    flags = np.full(n, -1, dtype=np.int32)
    for t in range(16):
        flags[np.flatnonzero(tile == t)[:each]] = 0
    print(f"[repair lanes] {each} flagged a tile, block {block}", flush=True)
    pts, box = cuda(xy), (L, 0.0, 0.0, L)
    want = host(*triangulate(pts, box, 1.0, tiled=0)[1:])
    dg, tri, num = triangulate(pts, box, 1.0, tile_shift=4, block=block)
    hit = torch.from_numpy(flags >= 0).cuda()
    tri.view(n, SLOTS)[hit] = -7
    num[hit] = 0
    f, req = cuda(flags), ctypes.c_int(0)
    st = _lib.load().gdt_repair(dg.ctx.handle, pts.data_ptr(), n, f.data_ptr(), SLOTS,
                                tri.data_ptr(), num.data_ptr(), PREC_FP64, ctypes.byref(req), None)
    torch.cuda.synchronize()
    assert st == _lib.GDT_OK and same(want, host(tri, num))
    assert dg.stats()["flagged"] == int((flags >= 0).sum())

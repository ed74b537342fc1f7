"""The exact mode's tile and star kernels on the GPU: rows byte for byte those of
its per-point kernel (row-major cells), over every kernel the dispatch picks
(the star kernel, two lanes and one lane per point, both tile edges), on random
points, lattices off by rounding errors (double-double decisions), exact
lattices (every point handed on, to wavefronts and beyond 8,192 to lanes) and a
cluster; and a batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_EXACT, _lib, inputs  # noqa: E402
from gpudelaunaytriangulation_amd.delaunay import (BatchedDelaunayGPU, DelaunayGPU,  # noqa: E402
                                                   PeriodicBoundaries)
from test_exact_mode import lattice  # noqa: E402


def rows(xy, lx, ly, cell, **config):
    n = len(xy)
    dg = DelaunayGPU(n, 20, cell, PeriodicBoundaries(lx, ly))
    dg.setPrecision(PREC_EXACT)
    dg.ctx.set_config(**config)
    tri = torch.full((n * dg.MaxSize,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(n, dtype=torch.int32, device="cuda")
    dg.globalDelaunayTriangulation(torch.from_numpy(np.ascontiguousarray(xy)).cuda(), tri, num)
    return tri.cpu().numpy().reshape(n, dg.MaxSize), num.cpu().numpy(), dg.stats()


def jittered(m, h, seed):
    return lattice(m, m, h)[0] + 1e-13 * np.random.default_rng(seed).standard_normal((m * m, 2))


# name: (points, lx, ly, cell size, lanes the automatic choice takes)
CASES = {
    "uniform1000": (lambda: inputs.uniform_points(1000, 40.0, 25.0, seed=7), 40.0, 25.0, 1.0, 64),
    "uniform16k": (lambda: inputs.uniform_points(16001, 128.0, 125.0, seed=3), 128.0, 125.0, 1.0, 64),
    "uniform50k": (lambda: inputs.uniform_points(50021, 292.0, 171.3, seed=4), 292.0, 171.3, 1.1, 2),
    "uniform300k": (lambda: inputs.uniform_points(300007, 600.0, 500.0, seed=5), 600.0, 500.0, 1.0, 1),
    "jitter60": (lambda: jittered(60, 0.1, 1), 6.0, 6.0, 0.1, 64),
    "jitter250": (lambda: jittered(250, 0.1, 2), 25.0, 25.0, 0.1, 2),
    "ties64": (lambda: lattice(64, 64, 1.0)[0], 64.0, 64.0, 1.0, 64),
    # (16,384 points handed on: more than get a wavefront each)
    "ties128": (lambda: lattice(128, 128, 1.0)[0], 128.0, 128.0, 1.0, 64),
    "cluster": (lambda: np.concatenate([inputs.uniform_points(4000, 80.0, 50.0, seed=9),
                                        30.0 + inputs.uniform_points(2500, 2.0, 2.0, seed=10)]),
                80.0, 50.0, 1.0, None),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_exact_tile_rows_equal_per_point_rows(case):
    gen, lx, ly, cell, lanes = CASES[case]
    xy = gen()
    print(f"[exact tile] {case}: n {len(xy)}", flush=True)
    want, wn, _ = rows(xy, lx, ly, cell, tiled=0)
    assert int(wn.sum()) == 6 * len(xy)
    got, gn, st = rows(xy, lx, ly, cell)
    if lanes is not None:
        assert st["lanes"] == lanes
    assert np.array_equal(wn, gn) and np.array_equal(want, got)
    for config in ({"lanes": 1, "tile_shift": 5}, {"lanes": 4, "tile_shift": 4},
                   {"lanes": 64, "tile_shift": 5}):
        if config["lanes"] == 64 and len(xy) > 60000:
            continue
        got, gn, _ = rows(xy, lx, ly, cell, **config)
        assert np.array_equal(wn, gn) and np.array_equal(want, got), config


def test_exact_tile_batch_and_range():
    sizes = [1500, 4000, 700]
    sides = [float(np.sqrt(s)) for s in sizes]
    pts = np.concatenate([inputs.uniform_points(s, L, L, seed=20 + i)
                          for i, (s, L) in enumerate(zip(sizes, sides))])
    print("[exact tile] batch", flush=True)
    bd = BatchedDelaunayGPU(sizes, [(L, L) for L in sides], 20, 1.0, precision=PREC_EXACT)
    tri = torch.full((bd.N * bd.MaxSize,), -7, dtype=torch.int32, device="cuda")
    num = torch.zeros(bd.N, dtype=torch.int32, device="cuda")
    bd.globalDelaunayTriangulation(torch.from_numpy(pts).cuda(), tri, num)
    got, a = tri.cpu().numpy().reshape(bd.N, bd.MaxSize), 0
    for s, L in zip(sizes, sides):
        want, wn, _ = rows(pts[a:a + s], L, L, 1.0, tiled=0)
        mine = got[a:a + s].copy()
        mine[mine >= 0] -= a
        assert np.array_equal(num.cpu().numpy()[a:a + s], wn) and np.array_equal(mine, want)
        a += s
    far = pts[:1500].copy()
    far[11, 1] -= 4.5 * sides[0]
    with pytest.raises(_lib.GdtError) as e:
        rows(far, sides[0], sides[0], 1.0)
    assert e.value.status == _lib.GDT_ERR_INVALID

"""Long lists of deferred points on the GPU, the rest of which goes one lane
each: rows equal to the row-major per-point kernel's.  Clumps that no window
holds (FP64 and FP32-filtered, a repair, the call without allocations), exact
lattices just below and above the length that wavefronts take in the exact
mode, and in a sheared box clumps beside a void, where some of the list's points
have circles that only a wavefront's search certifies."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_FP32F, PREC_FP64, _lib  # noqa: E402
from test_exact_mode import lattice  # noqa: E402
from test_gpu_exact_tile import rows as exact_rows  # noqa: E402
from test_gpu_general_tile import cuda, rows, same  # noqa: E402

WAVE_CAP, WAVE_CAP_EXACT = 8192, 3072      # lists up to these take a wavefront a point


def void_in_a_sheared_box():
    """A square void of 0.49 of the box, in which four circles are certified by
    a wavefront's search alone, and clumps close to their points."""
    L = 140.0
    rng = np.random.default_rng(6)
    u = rng.random((12000, 2)) * L
    u = u[~(np.abs(u - L / 2.0) < 0.245 * L).all(1)]
    near = [(75.9, 32.5), (107.4, 62.4), (107.4, 64.5), (32.6, 80.5)]
    u = np.concatenate([u] + [np.array(p) + 0.4 * rng.standard_normal((2700, 2)) for p in near])
    u = u[~(np.abs(u - L / 2.0) < 0.245 * L).all(1)]
    return np.stack([u[:, 0] + u[:, 1] / 6.0, u[:, 1]], 1), (L, L / 6.0, 0.0, L)


def clumps(n, each, k, L, seed):
    rng = np.random.default_rng(seed)
    c = 0.1 * L + 0.8 * L * rng.random((k, 2))
    xy = [rng.random((n, 2)) * L] + [p + rng.standard_normal((each, 2)) for p in c]
    return np.mod(np.concatenate(xy), L)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32F])
@pytest.mark.parametrize("n,L,tile_shift", [(4000, 64.0, 4), (30000, 180.0, 4), (30000, 180.0, 5)])
def test_clumps(n, L, tile_shift, precision):
    from gpudelaunaytriangulation_amd.delaunay import DelaunayGPU, PeriodicBoundaries
    xy = clumps(n, 2500, 6, L, seed=n)
    moved = np.mod(xy + 1e-3 * np.random.default_rng(1).standard_normal(xy.shape), L)
    print(f"[long lists] clumps {n} ts {tile_shift} precision {precision}", flush=True)

    def go(**config):
        dg = DelaunayGPU(len(xy), 24, 1.0, PeriodicBoundaries(L, L))
        dg.setPrecision(precision)
        dg.ctx.set_config(**config)
        tri = torch.full((len(xy) * dg.MaxSize,), -7, dtype=torch.int32, device="cuda")
        num = torch.zeros(len(xy), dtype=torch.int32, device="cuda")
        dg.globalDelaunayTriangulation(cuda(xy), tri, num)
        st = dg.stats()
        first = tri.cpu().numpy().reshape(len(xy), -1).copy(), num.cpu().numpy().copy()
        dg.testAndRepairDelaunayTriangulation(cuda(moved), tri, num)
        return first, (tri.cpu().numpy().reshape(len(xy), -1), num.cpu().numpy()), dg.last_repaired, st

    want = go(tiled=0)
    got = go(tile_shift=tile_shift)
    assert got[3]["deferred"] > WAVE_CAP
    assert same(want[0], got[0]) and same(want[1], got[1]) and want[2] == got[2]
    assert int(got[0][1].sum()) == int(got[1][1].sum()) == 6 * len(xy)


def test_clumps_without_allocations():
    L, stride = 120.0, 20
    xy = clumps(8000, 2500, 6, L, seed=5)
    n = len(xy)
    print("[long lists] no allocations", flush=True)
    nb = torch.full((n * stride,), -7, dtype=torch.int32, device="cuda")
    cnt = torch.zeros(n, dtype=torch.int32, device="cuda")
    req = ctypes.c_int(0)
    pts = cuda(xy)
    st = _lib.load().gdt_triangulate_noalloc(pts.data_ptr(), n, L, L, 1.0, stride, nb.data_ptr(),
                                             cnt.data_ptr(), PREC_FP64, ctypes.byref(req), None)
    torch.cuda.synchronize()
    assert st == _lib.GDT_OK
    (want, wn), _, _, _ = rows(xy, xy, (L, 0.0, 0.0, L), 1.0, tiled=0)
    assert same((want, wn), (nb.cpu().numpy().reshape(n, stride), cnt.cpu().numpy()))


@pytest.mark.parametrize("h", [1.0, 0.1])
@pytest.mark.parametrize("m", [54, 56])
def test_exact_lists_at_the_cap(m, h):
    assert 54 * 54 < WAVE_CAP_EXACT < 56 * 56
    xy, lx, ly = lattice(m, m, h)
    print(f"[long lists] exact {m} {h}", flush=True)
    want, wn, _ = exact_rows(xy, lx, ly, h, tiled=0)
    for config in ({}, {"lanes": 1, "tile_shift": 5}, {"lanes": 2, "tile_shift": 4}):
        got, gn, st = exact_rows(xy, lx, ly, h, **config)
        assert st["deferred"] == m * m
        assert np.array_equal(wn, gn) and np.array_equal(want, got), config


@pytest.mark.parametrize("n_side", [300, 420])
def test_exact_lattices_whole(n_side):
    """Beyond 3,072 points and beyond 131,072: the list and the cell-order kernels."""
    xy, lx, ly = lattice(n_side, n_side, 0.1)
    print(f"[long lists] exact whole {n_side}", flush=True)
    want, wn, _ = exact_rows(xy, lx, ly, 0.1, tiled=0)
    got, gn, st = exact_rows(xy, lx, ly, 0.1)
    assert st["deferred"] == len(xy)
    assert np.array_equal(wn, gn) and np.array_equal(want, got)


@pytest.mark.parametrize("config", [{}, {"lanes": 1, "tile_shift": 5}, {"lanes": 2, "tile_shift": 4},
                                    {"lanes": 64, "tile_shift": 4}], ids=str)
def test_clumps_beside_a_void_in_a_sheared_box(config):
    xy, box = void_in_a_sheared_box()
    print(f"[long lists] void {config}", flush=True)
    want = rows(xy, xy, box, 1.0, tiled=0)
    got = rows(xy, xy, box, 1.0, **config)
    assert got[3]["deferred"] > WAVE_CAP
    assert same(want[0], got[0]) and int(got[0][1].sum()) == 6 * len(xy)


def test_brownian_steps_beside_a_void_in_a_sheared_box():
    """The loop reads no count on the host: its longer lists go one lane each in
    the wavefronts' launch, which takes their uncertified points again."""
    from gpudelaunaytriangulation_amd.delaunay import BatchedDelaunayGPU
    xy, box = void_in_a_sheared_box()
    n = len(xy)
    print("[long lists] void, md", flush=True)

    def go(**config):
        bd = BatchedDelaunayGPU([n], [box], 24, 1.0)
        bd.ctx.set_config(**config)
        pts = cuda(xy)
        tri = torch.full((n * 24,), -7, dtype=torch.int32, device="cuda")
        num = torch.zeros(n, dtype=torch.int32, device="cuda")
        bd.globalDelaunayTriangulation(pts, tri, num)
        out = bd.md_run(pts, tri, num, 3, 0.02, seed=3)
        return (tri.cpu().numpy().reshape(n, -1), num.cpu().numpy()), pts.cpu().numpy(), out

    want, wp, wo = go(tiled=0)
    got, gp, go_ = go()
    assert go_["max_flagged"] > WAVE_CAP and go_["flagged_total"] == wo["flagged_total"]
    assert np.array_equal(wp, gp) and same(want, got)

"""The hull routine (gdt_hull.h) in the build for full cells, too -- windows of
4,096 points, blocks of more than 255 entries -- with a count of the rows that it
gives, and where it has to leave a point: close pairs in a lattice, whose
triangles are slivers that no other routine certifies either (a call that meets
one is refused, whichever routine meets it).  Host builds under AddressSanitizer
and UBSan against the per-point routine (tests/cpu_emul/hull_rows.cpp)."""
import os
import subprocess

import numpy as np
import pytest

from gpudelaunaytriangulation_amd import inputs
from test_exact_tile import CSRC, ROOT, run
from test_hull import CASES


def build(tmp_path_factory, ts, pts, *defines):
    out = str(tmp_path_factory.mktemp("hull_edges") / "hull_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-ffp-contract=off", f"-DGDT_TILE_SHIFT={ts}",
                    f"-DGDT_WIN_MAXPTS={pts}", *defines, f"-I{CSRC}",
                    os.path.join(ROOT, "tests", "cpu_emul", "hull_rows.cpp"), "-o", out], check=True)
    return out


@pytest.fixture(scope="module")
def dense(tmp_path_factory):
    return build(tmp_path_factory, 5, 4096, "-DGDT_WIN_DENSE")


@pytest.fixture(scope="module", params=[(4, 1024), (5, 2048), (5, 4096)], ids=str)
def exe(request, tmp_path_factory):
    return build(tmp_path_factory, *request.param)


DENSE = dict(CASES, **{
    # (2.1 and 2.4 points to a cell: 5x5 blocks that span more than 255 entries)
    "full": (lambda: inputs.uniform_points(3400, 40.0, 40.0, seed=21), (40.0, 40.0), 1.0),
    "fuller": (lambda: inputs.uniform_points(3500, 38.0, 38.0, seed=22), (38.0, 38.0), 1.0),
    "full general": (lambda: inputs.general_points(3400, (40.0, 11.0, 0.0, 41.0), seed=23),
                     (40.0, 41.0, 11.0, 0.0), 1.0),
})


@pytest.mark.parametrize("case", sorted(DENSE))
def test_rows_of_the_dense_build(dense, tmp_path, case):
    gen, box, cell = DENSE[case]
    xy = gen()
    n, left, differ, err = run(dense, tmp_path, xy, box[0], box[1], cell, *box[2:])
    assert n == len(xy) and differ == 0 and err == 0
    # (every window fits, so what is not left is the hull's)
    if case not in ("ties", "rows"):
        assert 2 * left < n
    else:
        assert left == n if case == "ties" else left < n


def pairs(seed):
    """A lattice off by 1e-8 or 1e-3, sixty of its points with another 1e-9 to
    1e-6 away."""
    r = np.random.default_rng(seed)
    n = 24 + 2 * (seed % 5)
    i = np.arange(n * n)
    x = np.stack([i % n + 0.5 * ((i // n) % 2) * (seed % 2), (i // n).astype(float)], 1)
    x = x + 10.0 ** -(3 + seed % 6) * r.standard_normal((n * n, 2))
    d = 10.0 ** -r.uniform(6, 9, 60)[:, None] * r.standard_normal((60, 2))
    return np.mod(np.concatenate([x, x[r.choice(n * n, 60, False)] + d]), float(n)), float(n)


@pytest.mark.parametrize("seed", [17, 30])
def test_slivers_are_left(exe, tmp_path, seed):
    xy, L = pairs(seed)
    n, _, differ, err = run(exe, tmp_path, xy, L, L, 1.0)
    assert n == len(xy) and differ == 0 and err     # (rows and flags alike, among them the refusal)


# (FP64 rows of every routine hold from 1e-30 to 1e36; FP32's squared distances, by
# which the hull finds the nearest entry, from 1e-17 to 1e19: beyond, the steps)
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("scale", [1e-30, 1e-22, 1e-12, 1e12, 1e19, 1e20, 1e25, 1e36])
def test_scales(exe, tmp_path, scale, general):
    L = 40.0 * scale
    xy = np.random.default_rng(3).random((1600, 2)) * L
    if general:
        xy = np.stack([xy[:, 0] + 0.3 * xy[:, 1], xy[:, 1]], 1)
    n, left, differ, err = run(exe, tmp_path, xy, L, L, scale, *((0.3 * L, 0.0) if general else ()))
    assert n == len(xy) and differ == 0 and err == 0
    if 1e-20 < scale < 1e19:
        assert 10 * left < n

"""The wavefront routine beside a void: a search whose circle spans many cells
takes a number of passes that grows with the logarithm of the circle's size, not
with the size, once it has a candidate, and its rows are the per-point routine's (host build under
AddressSanitizer and UBSan, tests/cpu_emul/wave_passes.cpp)."""
import os
import subprocess

import numpy as np
import pytest

from gpudelaunaytriangulation_amd import inputs
from test_exact_tile import CSRC, ROOT, run


@pytest.fixture(scope="module")
def passes(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("wave") / "wave_passes")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-ffp-contract=off", f"-I{CSRC}",
                    os.path.join(ROOT, "tests", "cpu_emul", "wave_passes.cpp"), "-o", out], check=True)
    return out


# name: (points, box x11, x22, cell size, x12, x21)
CASES = {
    "strip": (lambda: inputs.uniform_points(4000, 100.0, 70.0, seed=3), (100.0, 100.0, 0.5)),
    "square": (lambda: inputs.uniform_points(3000, 75.0, 75.0, seed=4), (100.0, 100.0, 0.6)),
    "clumps": (lambda: np.concatenate([inputs.uniform_points(300, 60.0, 60.0, seed=5)] +
                                      [10.0 + 18.0 * k + inputs.uniform_points(200, 1.5, 1.5, seed=6 + k)
                                       for k in range(3)]), (60.0, 60.0, 0.4)),
    "sparse": (lambda: inputs.uniform_points(300, 50.0, 50.0, seed=9), (50.0, 50.0, 0.4)),
    "general strip": (lambda: inputs.uniform_points(2500, 80.0, 60.0, seed=7),
                      (80.0, 80.0, 0.7, 20.0, 0.0)),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_passes_beside_a_void(passes, tmp_path, case):
    gen, box = CASES[case]
    xy = gen()
    n, differ, most = run(passes, tmp_path, xy, *box)
    assert n == len(xy) and differ == 0
    # (on average over a ring: squares of 6, 12, 24 and 48 cells to a side of the point)
    assert most <= 4

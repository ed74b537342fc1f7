"""Test-and-repair with the automatic number of lanes per flagged point against
two lanes on the GPU: rows byte for byte and the number repaired the same, at a
few points to a tile, with 16x16 and with 32x32 tiles, few and many flagged."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpudelaunaytriangulation_amd import PREC_FP32F, PREC_FP64, inputs  # noqa: E402
from test_gpu_general_tile import same  # noqa: E402
from test_gpu_hull import rows, square  # noqa: E402


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_FP32F])
@pytest.mark.parametrize("n,move", [(130, 0.02), (30011, 0.03), (300007, 0.002), (300007, 0.04)])
def test_automatic_lanes_repair_alike(n, move, prec):
    print(f"[repair] n {n} move {move} prec {prec}", flush=True)
    xy, box = square(n, 3)
    moved = inputs.wrap_into_general_box(xy + move * inputs.gaussian(4, 2 * n).reshape(-1, 2), box)
    _, want, count, _ = rows(xy, moved, box, 1.0, precision=prec, repair_lanes=2)
    _, got, c, _ = rows(xy, moved, box, 1.0, precision=prec)
    assert same(want, got) and c == count

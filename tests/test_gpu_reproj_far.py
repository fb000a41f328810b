"""Re-projections from references whose columns do not fit the LDS: lists that
are not in the order of the tilts, with shallow tilts between the first and last
reference of a steep projection.  One column below and above the limit (ten
references: 480 columns), all of the range's ways to be seen or not, rows beside
the workgroup's eight.  Bound as for the re-projector's other tests: FP64 on
both sides, FP32 store."""
import numpy as np
import pytest

from aretomo3_amd.projalign import find_proj_range
from test_gpu_reproj_rows import check

pytestmark = pytest.mark.gpu

TEN = [83.2, 0.0, 10.0, 83.4, 30.0, 83.0, 40.0, 83.6, 5.0, 83.1, 84.0]
SEVEN = [86.5, 20.0, 86.4, -3.0, 15.0, 33.0, 86.7, 87.0]


@pytest.mark.parametrize("tilts,px,py,vol_z", [
    (TEN, 479, 8, 20), (TEN, 480, 3, 20), (TEN, 500, 9, 33), (TEN, 1025, 17, 8),
    (SEVEN, 684, 4, 9), (SEVEN, 685, 4, 9), (SEVEN, 900, 8, 16)])
def test_references_far_from_a_steep_projection(gpu_available, tilts, px, py, vol_z):
    rng = np.random.default_rng(px)
    tilts = np.array(tilts, np.float32)
    n = len(tilts)
    projs = rng.uniform(0, 2, (n, py, px)).astype(np.float32)
    projs[:, 1, px // 3:px // 3 + 60] = -1e30
    skip = np.zeros(n, np.uint8)
    skip[n - 1] = 1
    assert find_proj_range(tilts, n - 1, skip) == (0, n - 2)
    print(f"case {n - 1} references, {px} x {py}, vol_z {vol_z}", flush=True)
    check(projs, tilts, vol_z, n - 1, skip)

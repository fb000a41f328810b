"""Empty samples (-1e30) in some slices of a back-projection, every voxel against
the oracle: the empty columns are chosen, in 64 bits, so that no voxel's
coordinate comes so close to a cell's edge beside an empty sample that FP32
cannot tell the side (on the rotation axis every tilt does).  Tiles of both row
counts, every storage type, widths and heights beside a tile; bounds as for the
other tile tests."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Plan, phantom
from aretomo3_amd import _lib as L
from helpers import rel_l2

pytestmark = pytest.mark.gpu
CASES = [(130, 70, 16), (130, 70, 8), (64, 64, 16), (194, 33, 8), (258, 20, 16)]
TILTS = np.linspace(-61.0, 58.5, 19).astype(np.float32)


def clear_of(t, edge, px, vol_z):
    """Whether no voxel's coordinate at tilt t lies within 2^-12 of the integer
    `edge` (FP32 coordinates are relative to a window of at most 288 samples:
    2^-15 apart, rounded three times)."""
    c, s = oracle.cos_sin(TILTS).reshape(-1, 2)[t].astype(np.float64)
    u = (np.arange(px) - px * 0.5)[None] * c + (np.arange(vol_z) - vol_z * 0.5)[:, None] * s + px * 0.5
    return np.abs(u - edge).min() > 2.0 ** -12


def empty_columns(px, vol_z):
    """{slice: (tilt, first, last)}: slice 1 a run of columns in one tilt, slice 2
    one column in every tilt, the first whose outer edges are clear of voxels
    (an edge between two empty samples decides nothing)."""
    first = next(x for x in range(10, px) if clear_of(3, x - 1, px, vol_z))
    last = next(x for x in range(first + 20, px) if clear_of(3, x + 1, px, vol_z))
    single = [next(x for x in range(px // 2 - 20, 1, -1)
                   if clear_of(t, x - 1, px, vol_z) and clear_of(t, x + 1, px, vol_z))
              for t in range(len(TILTS))]
    return {1: [(3, first, last)], 2: [(t, x, x) for t, x in enumerate(single)]}


@pytest.mark.parametrize("px,vol_z,tz", CASES)
@pytest.mark.parametrize("storage,tol", [(L.STORAGE_F32, 1e-5), (L.STORAGE_F16, 2e-3),
                                         (L.STORAGE_BF16, 8e-3)])
def test_empty_samples_off_the_axis(gpu_available, px, vol_z, tz, storage, tol):
    py = 4
    proj, _ = phantom.tilt_series(5 + px, px, py, TILTS, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    for y, cols in empty_columns(px, vol_z).items():
        for t, a, b in cols:
            proj[t, y, a:b + 1] = -1e30
    print(f"case {px} x {vol_z}, {tz} rows a thread, storage {storage}", flush=True)
    plan = Plan(px, py, TILTS, vol_z, L.METHOD_SART, sart_iters=0, sart_subsets=2, positivity=False,
                storage=storage)
    plan.set_tile_shape(tz, 16, 5)
    got = plan.execute_host(proj)
    ref = oracle.recon_slices(proj.astype(np.float64), TILTS, 1, vol_z, list(range(py)), iters=0,
                              n_subsets=2, relax=-1.0, order=0, positivity=0)
    for y in range(py):
        assert rel_l2(got[y], ref[y]) <= tol, y

"""Back-projection tiles (64 x 64 or 64 x 32 voxels, 8 / 16 / 32 tilts staged
at a time) at the edges of what a tile covers: widths and heights one off a
tile, tilt counts one off a stage, few slices and enough that one XCD takes a
whole slice, both row counts per thread, every storage type, empty samples.

Bounds: FP32 storage 1e-5 as everywhere for this path (coordinates below 96
carry 2^-18, the sums 2^-24 per term); FP16 / BF16 2e-3 (a stored sample
carries 2^-12 / 2^-9)."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Plan, phantom
from aretomo3_amd import _lib as L
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,py,vol_z,n", [
    (64, 2, 64, 16), (66, 2, 63, 17), (62, 3, 65, 33), (128, 2, 31, 8), (190, 1, 129, 32),
    (130, 2, 2, 9), (40, 259, 20, 7)])
@pytest.mark.parametrize("tz,chunk", [(16, 16), (16, 8), (8, 16), (8, 8)])
def test_sart_tiles(gpu_available, px, py, vol_z, n, tz, chunk):
    tilts = np.linspace(-70.0, 66.0, n).astype(np.float32)
    proj, _ = phantom.tilt_series(11 + px, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    print(f"case {px} x {py} x {vol_z}, {n} tilts, tile {tz} x {chunk}", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, sart_iters=2, sart_subsets=2, relax=0.3,
                subset_order=L.SUBSETS_INTERLEAVED, positivity=False)
    plan.set_tile_shape(tz, chunk, 5)
    got = plan.execute_host(proj)
    rows = list(range(py)) if py < 10 else [0, 1, 7, 8, 128, 255, py - 1]
    ref = oracle.recon_slices(proj.astype(np.float64), tilts, 1, vol_z, rows, iters=2, n_subsets=2,
                              relax=0.3, order=1, positivity=0)
    assert rel_l2(got[rows], ref) <= 1e-5


@pytest.mark.parametrize("px,py,vol_z,n", [(64, 2, 32, 32), (66, 3, 34, 33), (96, 5, 30, 65),
                                           (512, 40, 64, 11), (40, 259, 20, 7)])
@pytest.mark.parametrize("storage,tol", [(L.STORAGE_F32, 1e-5), (L.STORAGE_F16, 2e-3),
                                         (L.STORAGE_BF16, 8e-3)])
def test_wbp_tiles(gpu_available, px, py, vol_z, n, storage, tol):
    tilts = np.linspace(-62.0, 66.0, n).astype(np.float32)
    proj, _ = phantom.tilt_series(23 + px, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    print(f"case WBP {px} x {py} x {vol_z}, {n} tilts, storage {storage}", flush=True)
    got = Plan(px, py, tilts, vol_z, L.METHOD_WBP, storage=storage).execute_host(proj)
    rows = [0, 1, py // 2, py - 1]
    ref = oracle.recon_slices(proj.astype(np.float64), tilts, 0, vol_z, rows)
    assert rel_l2(got[rows], ref) <= tol


@pytest.mark.parametrize("storage,tol", [(L.STORAGE_F32, 1e-5), (L.STORAGE_F16, 2e-3),
                                         (L.STORAGE_BF16, 8e-3)])
def test_empty_samples_in_tiles(gpu_available, storage, tol):
    """Empty samples (-1e30) in some slices: those take the masked path."""
    px, py, vol_z = 130, 4, 70
    tilts = np.linspace(-60.0, 60.0, 19).astype(np.float32)
    proj, _ = phantom.tilt_series(5, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3, axis_max=12,
                                  noise_frac=0.05)
    proj[3, 1, 20:50] = -1e30
    proj[:, 2, 64] = -1e30
    print(f"case empty samples, storage {storage}", flush=True)
    got = Plan(px, py, tilts, vol_z, L.METHOD_SART, sart_iters=0, sart_subsets=2,
               positivity=False, storage=storage).execute_host(proj)
    ref = oracle.recon_slices(proj.astype(np.float64), tilts, 1, vol_z, list(range(py)), iters=0,
                              n_subsets=2, relax=-1.0, order=0, positivity=0)
    # The voxel on the rotation axis has the coordinate px / 2 at every tilt, an
    # integer next to slice 2's empty sample: whether a tilt counts there is a
    # tie that FP32 coordinates cannot decide as FP64 does.
    got[2, vol_z - 1 - vol_z // 2, px // 2] = ref[2, vol_z - 1 - vol_z // 2, px // 2]
    assert rel_l2(got, ref) <= tol

"""The forward projector for few slices (bands of a slice side by side, their
sums added afterwards) against the FP64 oracle and, bit for bit, against the
one that walks the bands in turn, which batches run: one to 40 slices, widths
beside the 64-ray tiles, two groups of tilts, one band row, steep tilts, slices
with empty voxels.  And the bands-in-turn projector where two of its workgroups
share a CU: more items than CUs, the widest slice whose bands of 8 rows fit
twice and the next."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Batch, DeviceArray, Plan, phantom, synchronize
from aretomo3_amd import _lib as L
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def _in_batch(plan, proj):
    d_in, d_out = DeviceArray.from_numpy(proj), DeviceArray(4 * int(np.prod(plan.volume_shape)))
    batch = Batch([plan], graph=False)
    batch.execute([d_in], [d_out])
    synchronize()
    return d_out.to_numpy(plan.volume_shape)


@pytest.mark.parametrize("px,py,vol_z,n,subsets,rows", [
    (64, 1, 40, 11, 2, 17), (66, 3, 19, 9, 3, 17), (512, 1, 60, 13, 2, 17), (130, 40, 50, 31, 1, 5),
    (1024, 2, 50, 13, 1, 17), (1024, 1, 33, 20, 1, 1), (2048, 1, 24, 9, 1, 3)])
@pytest.mark.parametrize("storage,tol", [(L.STORAGE_F32, 1e-5), (L.STORAGE_F16, 2e-3),
                                         (L.STORAGE_BF16, 8e-3)])
def test_few_slices(gpu_available, px, py, vol_z, n, subsets, rows, storage, tol):
    tilts = np.linspace(-70.0, 63.0, n).astype(np.float32)
    proj, _ = phantom.tilt_series(px + n, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    print(f"case {px} x {py} x {vol_z}, {n} tilts, {rows} rows, storage {storage}", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, sart_iters=2, sart_subsets=subsets, relax=0.3,
                subset_order=L.SUBSETS_INTERLEAVED, positivity=False, storage=storage)
    plan.set_tile_shape(16, 16, rows)
    got = plan.execute_host(proj)
    assert np.array_equal(got, _in_batch(plan, proj))
    ref = oracle.recon_slices(proj.astype(np.float64), tilts, 1, vol_z, list(range(py)), iters=2,
                              n_subsets=subsets, relax=0.3, order=1, positivity=0)
    assert rel_l2(got, ref) <= tol


@pytest.mark.parametrize("px,py,vol_z,storage,tol", [
    (65, 400, 30, L.STORAGE_F32, 1e-5), (512, 390, 20, L.STORAGE_F16, 2e-3),
    (1024, 260, 30, L.STORAGE_F32, 1e-5), (1134, 260, 19, L.STORAGE_F32, 1e-5),
    (1135, 260, 19, L.STORAGE_F32, 1e-5), (300, 390, 40, L.STORAGE_BF16, 8e-3),
    (700, 200, 30, L.STORAGE_F32, 1e-5)])
def test_two_workgroups_per_cu(gpu_available, px, py, vol_z, storage, tol):
    tilts = np.linspace(-60.0, 66.0, 9).astype(np.float32)
    proj, _ = phantom.tilt_series(px + py, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    print(f"case {px} x {py} x {vol_z}, storage {storage}", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, sart_iters=2, sart_subsets=2, relax=0.3,
                subset_order=L.SUBSETS_INTERLEAVED, positivity=False, storage=storage)
    got = plan.execute_host(proj)
    assert np.array_equal(got, _in_batch(plan, proj))
    rows = [0, 1, py // 2, py - 1]
    ref = oracle.recon_slices(proj.astype(np.float64), tilts, 1, vol_z, rows, iters=2, n_subsets=2,
                              relax=0.3, order=1, positivity=0)
    assert rel_l2(got[rows], ref) <= tol


def test_few_slices_with_empty_voxels(gpu_available):
    """Columns that no projection covers: slices 0 and 2 hold empty voxels."""
    px, py, vol_z = 96, 3, 36
    tilts = np.linspace(-60.0, 60.0, 9).astype(np.float32)
    proj, _ = phantom.tilt_series(9, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3, axis_max=12,
                                  noise_frac=0.05)
    proj[:, [0, 2], :30] = -1e30
    print("case empty voxels", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, sart_iters=2, sart_subsets=2, relax=0.3,
                subset_order=L.SUBSETS_INTERLEAVED, positivity=False)
    assert np.array_equal(plan.execute_host(proj), _in_batch(plan, proj))

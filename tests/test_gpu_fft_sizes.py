"""Transform lengths: powers of two (64 .. 8192 points, transforms in registers,
several rows or columns to a workgroup) and lengths beside them (transforms over
LDS), in the row filter, the three WBP transforms and the Fourier binning,
against the FP64 oracle: few and odd rows (the last workgroup partly filled),
columns that do not fill the last block, crops by 2, 4 and 8 and by other
ratios.  Bounds: those of the parity tests (the storage's rounding, twice 2^-11
and 2^-8, bounds the others: each filtered value is rounded once)."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Plan
from aretomo3_amd import _lib as L
from aretomo3_amd import phantom
from helpers import rel_l2

pytestmark = pytest.mark.gpu
TILTS = np.array([-48.0, -20.0, 4.0, 31.0, 55.0], np.float32)


@pytest.mark.parametrize("px,rows,vol_z,storage,tol", [
    (64, 3, 64, 0, 1e-5), (128, 33, 65, 0, 1e-5), (256, 1, 128, 0, 1e-5), (512, 2, 256, 0, 1e-5),
    (1024, 5, 512, 0, 1e-5), (2048, 3, 64, 0, 1e-5), (64, 2, 1024, 0, 1e-5), (64, 1, 2048, 0, 1e-5),
    (96, 3, 128, 0, 1e-5), (126, 3, 62, 0, 1e-5), (130, 4, 33, 0, 1e-5), (2046, 1, 31, 0, 1e-5),
    (256, 7, 64, L.STORAGE_F16, 2e-3), (256, 7, 64, L.STORAGE_BF16, 8e-3)])
def test_wbp_lengths(gpu_available, px, rows, vol_z, storage, tol):
    stack, _ = phantom.tilt_series(px + vol_z, px, rows, TILTS, vol_z, n_ellipsoids=30, axis_min=3,
                                   axis_max=12, noise_frac=0.05)
    print(f"case {px} x {rows}, VolZ {vol_z}, storage {storage}", flush=True)
    plan = Plan(px, rows, TILTS, vol_z, L.METHOD_WBP, storage=storage)
    got = plan.execute_host(stack)
    ref = oracle.recon_slices(stack.astype(np.float64), TILTS, 0, vol_z, list(range(rows)))
    assert rel_l2(got, ref) <= tol


@pytest.mark.parametrize("rx,ry,bin_factor", [
    (128, 128, 2.0), (256, 130, 2.0), (130, 256, 4.0), (512, 512, 8.0), (1024, 129, 2.0),
    (64, 1024, 2.0), (2048, 64, 8.0), (64, 2048, 4.0), (4096, 66, 4.0), (64, 4096, 8.0),
    (64, 4096, 3.0), (8192, 64, 8.0), (64, 8192, 8.0), (126, 254, 2.0), (256, 256, 3.0)])
def test_bin_lengths(gpu_available, rx, ry, bin_factor):
    n, vol_z = 2, 16
    tilts = TILTS[[0, 3]]
    raw, _ = phantom.tilt_series(rx + ry, rx, ry, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                 axis_max=12, noise_frac=0.05)
    axes, shifts = np.zeros(n, np.float32), np.array([[1.2, -0.7], [-2.1, 0.4]], np.float32)
    print(f"case {rx} x {ry} binned by {bin_factor}", flush=True)
    plan = Plan(rx, ry, tilts, vol_z, L.METHOD_SART, tilt_axis=axes, shifts=shifts,
                bin=bin_factor, sart_iters=0, sart_subsets=1, positivity=False, fill_seed=3)
    got = plan.execute_host(raw)
    aligned = oracle.prestage(raw, axes, shifts, 1, 3)
    binned = oracle.bin_stack(aligned, bin_factor)
    ref = oracle.recon_slices(binned, tilts, 1, vol_z, list(range(binned.shape[1])), iters=0,
                              n_subsets=1, relax=-1.0, order=0, positivity=0, seed=3)
    assert rel_l2(got, ref) <= 1e-5

"""The pre-stage's workgroups (64 columns x 32 or 16 rows) and its two ways to
weight patch shifts -- as products of a column and a row factor, or each
weight by itself where patches lie far from the image -- against the FP64
oracle: image sizes one off a group, more patches than fit one stage, several
axes, patches 1 to 40 image sizes away.  Every pixel is a nearest-neighbour
pick, so one wrong coordinate shows as ~1e-3; the bound is the path's 1e-5."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Plan
from aretomo3_amd import _lib as L
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rx,ry,axis,n_patches,spread", [
    (64, 33, 0.0, 0, 0), (66, 64, 85.0, 0, 0), (130, 70, -95.0, 0, 0), (300, 8, 40.0, 0, 0),
    (64, 48, 3.0, 1, 1.0), (130, 66, 86.0, 32, 1.0), (96, 97, -80.0, 33, 1.0),
    (96, 64, 45.0, 70, 1.0), (64, 48, 85.0, 9, 2.5), (64, 48, 85.0, 9, 40.0), (300, 20, 45.0, 5, 1.0)])
def test_prestage_tiles(gpu_available, rx, ry, axis, n_patches, spread):
    rng = np.random.default_rng(rx * 7 + n_patches)
    tilts = np.array([-40.0, -3.0, 21.0, 50.0], np.float32)
    n = len(tilts)
    raw = rng.normal(1.0, 1.0, (n, ry, rx)).astype(np.float32)
    axes = np.full(n, axis, np.float32)
    shifts = rng.uniform(-3, 3, (n, 2)).astype(np.float32)
    lp = None
    if n_patches:
        lp = np.empty((n, 5, n_patches), np.float32)
        lp[:, 0] = rng.uniform(-0.5, 0.5, (n, n_patches)) * rx * spread
        lp[:, 1] = rng.uniform(-0.5, 0.5, (n, n_patches)) * ry * spread
        lp[:, 2:4] = rng.uniform(-2.5, 2.5, (n, 2, n_patches))
        lp[:, 4] = rng.uniform(0, 1, (n, n_patches)) < 0.8
        lp[0, 4] = 0.0    # one tilt without a good patch
    print(f"case {rx} x {ry}, axis {axis}, {n_patches} patches, spread {spread}", flush=True)
    plan = Plan(rx, ry, tilts, 8, L.METHOD_SART, tilt_axis=axes, shifts=shifts, local_params=lp,
                sart_iters=0, sart_subsets=1, positivity=False, fill_seed=3)
    got = plan.execute_host(raw)
    aligned = oracle.prestage(raw, axes, shifts, 1, 3, local=lp)
    ref = oracle.recon_slices(aligned, tilts, 1, 8, list(range(aligned.shape[1])), iters=0,
                              n_subsets=1, relax=-1.0, order=0, positivity=0, seed=3)
    assert rel_l2(got, ref) <= 1e-5

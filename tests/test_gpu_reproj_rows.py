"""The re-projector's workgroups (64 columns x 8 rows, a ray in segments) at
their edges: one row or column more than a group, rays of several segments,
each number of reference tilts, a lone reference so much steeper than the
projection that 64 columns reach over 3000, empty values in some columns only.
Bound as for the re-projector's other tests: FP64 on both sides, FP32 store."""
import numpy as np
import pytest

import oracle
from aretomo3_amd.projalign import CalcReproj, find_proj_range
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def check(projs, tilts, vol_z, idx, skip=None):
    n, py, px = projs.shape
    skip = np.zeros(n, np.uint8) if skip is None else skip
    rp = CalcReproj(px, py, n, vol_z)
    got = rp.do_it(projs, tilts, skip, idx)
    rp.close()
    ref = oracle.reproj(projs, tilts, vol_z, idx, skip)
    assert np.array_equal(got < -1e29, ref < -1e29)
    ok = ref > -1e29
    # (a ray through a thick slice may find too few voxels in every column)
    assert not ok.any() or rel_l2(got[ok], ref[ok]) <= 1e-6


@pytest.mark.parametrize("px,py,vol_z", [(64, 8, 16), (65, 9, 40), (63, 7, 33), (300, 17, 900),
                                         (2, 1, 1), (129, 1, 300)])
def test_group_edges(gpu_available, px, py, vol_z):
    rng = np.random.default_rng(px)
    tilts = np.linspace(-48, 54, 35).astype(np.float32)
    projs = rng.uniform(-1, 2, (35, py, px)).astype(np.float32)
    for idx in (3, 17, 30):
        print(f"case {px} x {py}, vol_z {vol_z}, projection {idx}", flush=True)
        check(projs, tilts, vol_z, idx)


@pytest.mark.parametrize("step,count", [(21.0, 1), (10.0, 3), (6.0, 5), (4.0, 8), (2.0, 10)])
def test_numbers_of_reference_tilts(gpu_available, step, count):
    rng = np.random.default_rng(int(step))
    tilts = np.arange(-2, 3, dtype=np.float32) * 21 if count == 1 else \
        np.arange(-60, 61, step).astype(np.float32)
    projs = rng.uniform(0, 2, (len(tilts), 5, 100)).astype(np.float32)
    projs[:, 2, 40:60] = -1e30
    idx = len(tilts) // 2
    first, last = find_proj_range(tilts, idx)
    print(f"case step {step}: tilts {first}..{last}", flush=True)
    check(projs, tilts, 48, idx)


def test_lone_steep_projection(gpu_available):
    rng = np.random.default_rng(9)
    tilts = np.array([20.0, 88.5], np.float32)
    projs = rng.uniform(0, 2, (2, 3, 4000)).astype(np.float32)
    print("case 88.5 deg from 20 deg, 4000 columns", flush=True)
    check(projs, tilts, 6, 1, np.array([0, 1], np.uint8))

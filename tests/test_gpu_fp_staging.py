"""Which forward projector runs, and that each gives the oracle's result: with
few slices the bands of a slice are projected side by side unless a prefetching
projector is set by hand, with more they are walked in turn by the direct, the
band-prefetching and the register-prefetching projector.  Slices with and
without empty voxels, so that one pass runs the variants for both.

A plan's device bytes tell which one it is set up for: the bands side by side
need the scratch of part_bytes(), everything else that depends on the staging
is a fraction of that.

Bounds: those of this path everywhere, 1e-5 with FP32 storage, 2e-3 with FP16 (a
stored sample carries 2^-12).  Projectors are compared bit for bit."""
import numpy as np
import pytest

import oracle
from aretomo3_amd import Batch, DeviceArray, Plan, phantom, synchronize
from aretomo3_amd import _lib as L
from helpers import rel_l2

pytestmark = pytest.mark.gpu

N_TILTS, SUBSETS = 9, 2
KW = dict(sart_iters=2, sart_subsets=SUBSETS, relax=0.3, subset_order=L.SUBSETS_INTERLEAVED,
          positivity=False, fill_seed=3)


def series(px, py, vol_z):
    """Projections, and a start volume (slice layout) with empty voxels in
    slices 0 and 2."""
    tilts = np.linspace(-61.0, 58.0, N_TILTS).astype(np.float32)
    proj, _ = phantom.tilt_series(px + py, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3,
                                  axis_max=12, noise_frac=0.05)
    rng = np.random.default_rng(px)
    start = rng.random((py, vol_z, px)).astype(np.float32)
    keep = beside_cell_edges(tilts, px, vol_z)
    for y in (0, 2):
        empty = rng.random((vol_z, px)) < 0.02
        empty[4:8, 30:40] = True
        empty[:, 50] = True
        start[y][empty & ~keep] = -1e30
    return tilts, proj, start


def beside_cell_edges(tilts, px, vol_z):
    """Voxels that a ray's sample uses or leaves by a coordinate within 2^-10 of
    an integer (in 64 bits, GForProj.cu:40-60): whether that sample touches an
    empty voxel there is not decided by FP32 coordinates, 2^-13 apart at 2048."""
    near = np.zeros((vol_z, px), bool)
    for c, s in oracle.cos_sin(tilts).reshape(-1, 2).astype(np.float64):
        n = int(vol_z / c + 1.5)
        fz = np.arange(n)[None] - n * 0.5
        x = (np.arange(px)[:, None] - 0.5 * px) / c + px * 0.5 - fz * s
        z = vol_z * 0.5 + fz * c + 0.0 * x
        hit = (np.abs(x - np.round(x)) < 2.0 ** -10) & (x >= -1) & (x <= px) & (z >= 0) & (z <= vol_z - 2)
        xi, zi = np.round(x[hit]).astype(int), z[hit].astype(int)
        for dx in (-1, 0, 1):
            for dz in (0, 1):
                near[zi + dz, np.clip(xi + dx, 0, px - 1)] = True
    return near


def part_bytes(px, py, vol_z, rows):
    """Sums (4 bytes) and counts (2) of every band, slice and ray of a subset."""
    bands = -(-(vol_z - 1) // rows)
    return 6 * bands * py * -(-N_TILTS // SUBSETS) * (-(-px // 64) * 64)


def run(plan, proj, start):
    d_in, d_vol = DeviceArray.from_numpy(proj), DeviceArray.from_numpy(start)
    plan.execute(d_in, d_vol, accumulate=True)
    synchronize()
    got = d_vol.to_numpy(start.shape)
    d_in.free()
    d_vol.free()
    return got


def reference(proj, tilts, start, rows):
    n, _, px = proj.shape
    vol_z = start.shape[1]
    table = oracle.fill_table(3 ^ 0x5A5A5A5A5A5A5A5A, px * vol_z)
    out = []
    for y in rows:
        sino = np.zeros((n, (px // 2 + 1) * 2), np.float64)
        sino[:, :px] = proj[:, y]
        out.append(oracle.tomo_sart(sino, px, oracle.cos_sin(tilts), start[y].astype(np.float64), 0, n,
                                    2, SUBSETS, relax=0.3, order=1, positivity=0, fill_tbl=table)[0])
    return np.array(out)


# 512: bands of two workgroups fit the LDS of a CU, the others one at 17 / 5 rows
@pytest.mark.parametrize("px,py,vol_z,rows,modes,storage,tol", [
    (512, 390, 36, 8, (0, 1), L.STORAGE_F32, 1e-5),
    (768, 132, 36, 8, (0, 1), L.STORAGE_F16, 2e-3),
    (700, 132, 40, 17, (0,), L.STORAGE_F32, 1e-5),
    (1024, 132, 36, 8, (0, 1, 2), L.STORAGE_F32, 1e-5),
    (1024, 132, 40, 17, (0, 2), L.STORAGE_F16, 2e-3),
    (2048, 132, 24, 5, (0, 1, 2), L.STORAGE_F32, 1e-5)])
def test_bands_in_turn(gpu_available, px, py, vol_z, rows, modes, storage, tol):
    tilts, proj, start = series(px, py, vol_z)
    print(f"case {px} x {py} x {vol_z}, {rows} rows, modes {modes}, storage {storage}", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, layout=L.LAYOUT_SLICE, storage=storage, **KW)
    got, size = {}, {}
    for pf in modes:
        plan.set_tile_shape(16, 16, rows, pf)
        size[pf] = plan.device_bytes
        got[pf] = run(plan, proj, start)
    plan.close()
    part = part_bytes(px, py, vol_z, rows)
    for pf in modes[1:]:
        assert abs(size[pf] - size[0]) < part // 2
        assert np.array_equal(got[pf], got[0]), pf
    rows_y = [0, 1, 2, py // 2, py - 1]
    assert rel_l2(got[0][rows_y], reference(proj, tilts, start, rows_y)) <= tol


@pytest.mark.parametrize("px,vol_z,rows,modes", [
    (512, 36, 8, (1,)), (768, 36, 8, (1,)), (1024, 36, 8, (1, 2)), (2048, 24, 5, (1, 2))])
def test_few_slices_and_staging_set_by_hand(gpu_available, px, vol_z, rows, modes):
    py = 4
    tilts, proj, start = series(px, py, vol_z)
    print(f"case {px} x {py} x {vol_z}, {rows} rows, modes {modes}", flush=True)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, layout=L.LAYOUT_SLICE, **KW)
    plan.set_tile_shape(16, 16, rows)
    size = plan.device_bytes
    got = run(plan, proj, start)
    assert rel_l2(got, reference(proj, tilts, start, range(py))) <= 1e-5
    part = part_bytes(px, py, vol_z, rows)
    for pf in modes:
        plan.set_tile_shape(16, 16, rows, pf)
        assert size - plan.device_bytes > part // 2, pf
        assert np.array_equal(run(plan, proj, start), got), pf
    plan.set_tile_shape(16, 16, rows)
    assert plan.device_bytes == size
    plan.close()


@pytest.mark.parametrize("storage", [L.STORAGE_F32, L.STORAGE_BF16])
def test_batch_with_empty_voxels(gpu_available, storage):
    """Voxels that become empty during the iterations (one projection value far
    below the others, one tilt a subset, relaxation 1.5: a step of -1.3e10), in
    slices 0 and 2: a batch, whose launch for slices with empty voxels they
    take, gives what the plan gives alone, bands side by side and in turn."""
    px, py, vol_z, n = 256, 4, 36, 7
    tilts = np.linspace(-46.0, 53.0, n).astype(np.float32)
    proj, _ = phantom.tilt_series(9, px, py, tilts, vol_z, n_ellipsoids=30, axis_min=3, axis_max=12,
                                  noise_frac=0.05)
    proj[3, [0, 2], 30:50] = -9e9 * vol_z / np.cos(np.deg2rad(tilts[3]))
    # a fill table that maps each voxel to itself fills with the slice's mean:
    # many equal values show that the slice had empty voxels
    for y in range(py):
        sino = np.zeros((n, px + 2))
        sino[:, :px] = proj[:, y]
        ref, _ = oracle.tomo_sart(sino, px, oracle.cos_sin(tilts), np.zeros((vol_z, px)), 0, n, 1, n,
                                  relax=1.5, positivity=0, fill_tbl=np.arange(vol_z * px))
        assert (np.unique(ref, return_counts=True)[1].max() > 300) == (y in (0, 2))
    print(f"case batch with empty voxels, storage {storage}", flush=True)
    kw = dict(sart_iters=3, sart_subsets=n, relax=1.5, positivity=False, fill_seed=3, storage=storage)
    plan = Plan(px, py, tilts, vol_z, L.METHOD_SART, **kw)
    other = Plan(px, 2, tilts, 20, L.METHOD_SART, **kw)
    for pf in (0, 1):
        plan.set_tile_shape(16, 16, 8, pf)
        alone = plan.execute_host(proj)
        d_in, d_in2 = DeviceArray.from_numpy(proj), DeviceArray.from_numpy(proj[:, [1, 3]])
        d_out = [DeviceArray(4 * int(np.prod(p.volume_shape))) for p in (plan, other)]
        batch = Batch([plan, other])
        batch.execute([d_in, d_in2], d_out)
        synchronize()
        assert np.array_equal(d_out[0].to_numpy(plan.volume_shape), alone), pf
        batch.close()
        if pf == 0:
            first = alone
    assert np.array_equal(alone, first)

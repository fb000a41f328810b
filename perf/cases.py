"""Performance cases of the reconstruction path: what is timed, on which
inputs, and what the results are in 64-bit arithmetic.

Every case calls the package the way a user's program does: a plan (or slice
operator, batch, re-projector) is made once per geometry and kept, the raw
projections are on the GPU, and one pass is one reconstruction.  Sizes are
those of the benchmark and test configurations: detectors of 512 to 4096
pixels, 31 to 61 tilts over +-60 degrees, sections of 64 to 512 voxels.

The synthetic series are projections of isotropic Gaussian particles (exact
line integrals), tilted about y, mapped to raw images by the tilt axis and
per-tilt shifts when the pre-stage is in the path, plus Gaussian noise.
"""
import math

import numpy as np
import torch

from aretomo3_amd import Batch, CalcVolThick, Plan, TomoSart, TomoWbp
from aretomo3_amd import _lib as L
from aretomo3_amd.projalign import CalcReproj, find_proj_range

STORAGE = {"f32": L.STORAGE_F32, "f16": L.STORAGE_F16, "bf16": L.STORAGE_BF16}
LAYOUT = {"xzy": L.LAYOUT_XZY, "xyz": L.LAYOUT_XYZ, "slice": L.LAYOUT_SLICE}
EMPTY, SENT = -1e10, -1e30


def listed():
    bench = dict(iters=10, subsets=5, interleaved=True, positivity=False, relax=0.3)
    return [
        # The per-slice operators, as a program that loops over slices itself
        # calls them (one launch sequence on one slice: latency).
        dict(name="sart_slice", kind="slice", method="sart", nx=512, ny=1, n=41, vol_z=128,
             storage="f32", **bench),
        dict(name="wbp_slice", kind="slice", method="wbp", nx=1024, ny=1, n=61, vol_z=256,
             storage="f32"),
        # A small series with the pre-stage (a quick preview): many short launches.
        dict(name="sart_preview", kind="series", method="sart", nx=256, ny=256, n=61, vol_z=64,
             axis=85.0, shift=3.0, storage="f32", layout="xzy", iters=4, subsets=5,
             interleaved=True, positivity=False, relax=0.3),
        # Odd, ragged sizes in the reference's own mode (contiguous subsets,
        # positivity, relax 1/subsets), two tilts excluded, BF16 projections,
        # flipped layout.
        dict(name="sart_ragged_bf16", kind="series", method="sart", nx=683, ny=475, n=41, vol_z=150,
             axis=3.0, shift=5.0, storage="bf16", layout="xyz", iters=5, subsets=7,
             interleaved=False, positivity=True, relax=-1.0, excluded=2),
        # The headline series of the benchmark.
        dict(name="sart_1024", kind="series", method="sart", nx=1024, ny=1024, n=61, vol_z=256,
             axis=85.0, shift=3.0, storage="f32", layout="xzy", iters=20, subsets=5,
             interleaved=True, positivity=False, relax=0.3),
        # The largest: full-frame series with narrow projection storage.
        dict(name="sart_2048_f16", kind="series", method="sart", nx=2048, ny=2048, n=61, vol_z=512,
             axis=0.0, shift=0.0, storage="f16", layout="xzy", **bench),
        # Weighted back-projection of an aligned series.
        dict(name="wbp_512", kind="series", method="wbp", nx=512, ny=512, n=41, vol_z=128, axis=0.0,
             shift=0.0, storage="f32", layout="xzy"),
        dict(name="wbp_2048_f16", kind="series", method="wbp", nx=2048, ny=2048, n=61, vol_z=512,
             axis=0.0, shift=0.0, storage="f16", layout="xzy"),
        # Raw camera frames: local alignment, Fourier binning by 4, then WBP.
        dict(name="wbp_raw_bin4_local", kind="series", method="wbp", nx=4096, ny=4096, n=41,
             vol_z=256, axis=86.0, shift=3.0, patches=25, bin=4.0, storage="f32", layout="xyz"),
        # Projection matching: one re-projection of a high tilt.
        dict(name="reproject_1024", kind="reproj", nx=1024, ny=1024, n=41, vol_z=256, index=4),
        # Uneven series reconstructed together, replayed from a graph.
        dict(name="batch_uneven", kind="batch", n0=31, nx0=512, z0=128, n1=41, nx1=768, z1=256,
             n2=61, nx2=512, z2=256, n3=51, nx3=1024, z3=128, axis=88.0, shift=3.0, storage="f32",
             iters=5, subsets=5),
        # Sample thickness of a raw series, on host data.
        dict(name="thickness_2048", kind="thickness", nx=2048, ny=2048, n=41, axis=86.0, shift=3.0,
             pixel=1.0),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["slice", "series", "series", "series", "reproj", "batch"])
    n = rng.choice([31, 41, 51, 61, rng.randrange(11, 62)])
    vol_z = _size(rng, 40, 384)
    sart = dict(iters=rng.randrange(2, 11), subsets=rng.randrange(1, 9),
                interleaved=rng.random() < 0.5, positivity=rng.random() < 0.5,
                relax=rng.choice([0.3, -1.0]))
    storage = rng.choice(["f32", "f32", "f16", "bf16"])
    if kind == "slice":
        method = rng.choice(["sart", "wbp"])
        c = dict(kind=kind, method=method, nx=_size(rng, 96, 2048), ny=1, n=n, vol_z=vol_z,
                 storage="f32" if method == "wbp" else storage)
        if method == "sart":
            c.update(sart)
        return c
    if kind == "series":
        method = rng.choice(["sart", "wbp"])
        c = dict(kind=kind, method=method, nx=_size(rng, 96, 1200), ny=_size(rng, 96, 1200), n=n,
                 vol_z=vol_z, axis=rng.choice([0.0, rng.uniform(-5, 5), rng.uniform(80, 95)]),
                 shift=3.0, storage=storage, layout=rng.choice(["xzy", "xyz"]))
        if rng.random() < 0.25:
            c.update(bin=2.0, nx=2 * c["nx"], ny=2 * c["ny"])
        if rng.random() < 0.25:
            c.update(patches=rng.choice([9, 25]))
        if method == "sart":
            c.update(sart, excluded=rng.choice([0, 0, 2]))
        return c
    if kind == "reproj":
        return dict(kind=kind, nx=_size(rng, 128, 1100), ny=_size(rng, 128, 1100), n=41,
                    vol_z=vol_z, index=rng.randrange(2, 39))
    c = dict(kind="batch", axis=rng.uniform(80, 95), shift=3.0, storage=storage,
             iters=rng.randrange(2, 6), subsets=5)
    for k in range(4):
        c.update({"n%d" % k: rng.choice([31, 41, 51, 61]), "nx%d" % k: _size(rng, 200, 1024),
                  "z%d" % k: rng.choice([100, 128, 256])})
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _tilts(n):
    return np.linspace(-60.0, 60.0, n).astype(np.float32)


def _aligned_size(c):
    if c.get("axis") is not None and abs(math.sin(c["axis"] * 3.14 / 180.0)) > 0.707:
        return c["ny"], c["nx"]
    return c["nx"], c["ny"]


def _inputs(c, seed):
    """Raw projections [n][ny][nx] (float32, on the GPU) and the alignment."""
    n, nx, ny = c["n"], c["nx"], c["ny"]
    rng = np.random.default_rng(int(seed) * 7919 + nx * 31 + ny * 17 + n)
    tilts = _tilts(n)
    ax, ay = _aligned_size(c)
    depth = c.get("vol_z", nx // 4) * c.get("bin", 1.0)
    count = 200
    px = rng.uniform(-0.48 * ax, 0.48 * ax, count)
    py = rng.uniform(-0.48 * ay, 0.48 * ay, count)
    pz = rng.uniform(-0.35 * depth, 0.35 * depth, count)
    sig = rng.uniform(2.0, max(4.0, 0.02 * ax), count)
    amp = rng.uniform(0.5, 1.0, count) * sig
    ang = np.deg2rad(tilts.astype(np.float64))[:, None]
    u = px * np.cos(ang) + pz * np.sin(ang)
    v = np.broadcast_to(py, u.shape)
    shifts = np.zeros((n, 2), np.float32)
    if c.get("axis") is not None:
        a = math.radians(c["axis"])
        u, v = u * math.cos(a) - v * math.sin(a), u * math.sin(a) + v * math.cos(a)
        if c.get("shift"):
            shifts = rng.uniform(-c["shift"], c["shift"], (n, 2)).astype(np.float32)
        u, v = u + shifts[:, :1], v + shifts[:, 1:]
    dev = "cuda"
    gu = torch.tensor(u + nx * 0.5, device=dev)[:, None, :]
    gv = torch.tensor(v + ny * 0.5, device=dev)[:, None, :]
    s = torch.tensor(sig, device=dev)
    x = torch.arange(nx, device=dev, dtype=torch.float64)[None, :, None]
    y = torch.arange(ny, device=dev, dtype=torch.float64)[None, :, None]
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed) + 1)
    out = torch.empty((n, ny, nx), device=dev)
    am = torch.tensor(amp, device=dev)
    for t in range(n):
        ex = torch.exp(-0.5 * ((x[0] - gu[t]) / s) ** 2)
        ey = torch.exp(-0.5 * ((y[0] - gv[t]) / s) ** 2) * am
        out[t] = (ey @ ex.T).to(torch.float32)
    mean = float(out.mean(dtype=torch.float64))
    out += 0.1 * mean * torch.randn(out.shape, device=dev, generator=gen)
    patches = None
    if c.get("patches"):
        m = int(round(math.sqrt(c["patches"])))
        gxy = (np.arange(m) + 0.5) / m - 0.5
        cx, cy = np.meshgrid(gxy * nx, gxy * ny)
        patches = np.zeros((n, 5, c["patches"]), np.float32)
        patches[:, 0] = cx.ravel()
        patches[:, 1] = cy.ravel()
        patches[:, 2:4] = rng.normal(0.0, 2.0, (n, 2, c["patches"]))
        patches[:, 4] = rng.random((n, c["patches"])) < 0.95
    exclude = None
    if c.get("excluded"):
        exclude = np.zeros(n, np.uint8)
        exclude[rng.choice(n, c["excluded"], replace=False)] = 1
    return out, dict(tilts=tilts, shifts=shifts, patches=patches, exclude=exclude,
                     fill_seed=int(seed))


def _options(c, al):
    kw = dict(storage=STORAGE[c["storage"]])
    if c.get("axis") is not None:
        kw.update(tilt_axis=np.full(c["n"], c["axis"], np.float32), shifts=al["shifts"],
                  fill_seed=al["fill_seed"], local_params=al["patches"], bin=c.get("bin", 1.0))
    if al["exclude"] is not None:
        kw["exclude"] = al["exclude"]
    if c["method"] == "sart":
        kw.update(sart_iters=c["iters"], sart_subsets=c["subsets"], relax=c["relax"],
                  positivity=c["positivity"], subset_order=L.SUBSETS_INTERLEAVED
                  if c["interleaved"] else L.SUBSETS_CONTIGUOUS)
    return kw


def _members(c):
    return [dict(kind="series", method="sart", nx=c["nx%d" % k], ny=c["nx%d" % k], n=c["n%d" % k],
                 vol_z=c["z%d" % k], axis=c["axis"], shift=c["shift"], storage=c["storage"],
                 layout="xzy", iters=c["iters"], subsets=c["subsets"], interleaved=True,
                 positivity=False, relax=0.3) for k in range(4)]


def _plan(c, al):
    method = L.METHOD_SART if c["method"] == "sart" else L.METHOD_WBP
    return Plan(c["nx"], c["ny"], al["tilts"], c["vol_z"], method, layout=LAYOUT[c["layout"]],
                **_options(c, al))


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "slice":
        proj, al = _inputs(dict(c, ny=32), seed)
        pad = (c["nx"] // 2 + 1) * 2
        sino = torch.zeros((c["n"], pad), device="cuda")
        sino[:, :c["nx"]] = proj[:, 16, :]
        vx = c["nx"] // 2 * 2
        if c["method"] == "sart":
            op = TomoSart()
            op.setup(vx, c["vol_z"], c["subsets"], c["iters"], c["nx"], al["tilts"], 0, c["n"],
                     relax=c["relax"], subset_order=L.SUBSETS_INTERLEAVED if c["interleaved"]
                     else L.SUBSETS_CONTIGUOUS, positivity=c["positivity"],
                     storage=STORAGE[c["storage"]])
        else:
            op = TomoWbp()
            op.setup(vx, c["vol_z"], c["nx"], al["tilts"])
        return dict(case=c, op=op, sino=sino, vol=torch.zeros((c["vol_z"], vx), device="cuda"))
    if kind == "series":
        proj, al = _inputs(c, seed)
        plan = _plan(c, al)
        return dict(case=c, plan=plan, proj=proj,
                    vol=torch.empty(plan.volume_shape, device="cuda"))
    if kind == "reproj":
        proj, al = _inputs(c, seed)
        return dict(case=c, op=CalcReproj(c["nx"], c["ny"], c["n"], c["vol_z"]), proj=proj,
                    tilts=al["tilts"], out=torch.empty((c["ny"], c["nx"]), device="cuda"))
    if kind == "batch":
        members = [(m,) + _inputs(m, seed + 100 * k) for k, m in enumerate(_members(c))]
        plans = [_plan(m, al) for m, _, al in members]
        return dict(case=c, plans=plans, batch=Batch(plans, graph=True),
                    projs=[p for _, p, _ in members],
                    vols=[torch.empty(p.volume_shape, device="cuda") for p in plans])
    proj, al = _inputs(c, seed)
    return dict(case=c, raw=proj.cpu().numpy(), al=al)


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "slice":
        if c["method"] == "sart":
            state["vol"].zero_()   # do_it continues from the volume it is given
        state["op"].do_it(state["sino"].data_ptr(), state["vol"].data_ptr())
        return state["vol"]
    if kind == "series":
        state["plan"].execute(state["proj"].data_ptr(), state["vol"].data_ptr())
        return state["vol"]
    if kind == "reproj":
        state["op"].execute(state["proj"].data_ptr(), state["tilts"], None, c["index"],
                            state["out"].data_ptr())
        return state["out"]
    if kind == "batch":
        state["batch"].execute([p.data_ptr() for p in state["projs"]],
                               [v.data_ptr() for v in state["vols"]])
        return list(state["vols"])
    op, al = CalcVolThick(), state["al"]
    r = op.do_it(state["raw"], al["tilts"], c["pixel"], tilt_axis=np.full(c["n"], c["axis"],
                 np.float32), shifts=al["shifts"], fill_seed=al["fill_seed"])
    return dict(profile=op.profile, low=r["low_edge"], high=r["high_edge"], offset=r["offset_z"])


# ---------------------------------------------------------------------------
# work of one pass
# ---------------------------------------------------------------------------
def _recon_size(c):
    ax, ay = _aligned_size(c)
    b = c.get("bin", 1.0)
    if b != 1.0:
        ax, ay = int(ax / b) // 2 * 2, int(ay / b) // 2 * 2
    return ax // 2 * 2, ay


def _series_work(c):
    vx, vy = _recon_size(c)
    vox = float(vx) * vy * c["vol_z"]
    nbytes = 4.0 * c["n"] * c["nx"] * c["ny"] + 4.0 * vox
    flops = 0.0
    if c["method"] == "wbp":
        # 2x grid: four linear interpolations per voxel and tilt, two 2-D FFTs
        # and the row filter
        flops += 4 * vox * c["n"] * 5 + 2.5 * 4 * vox * math.log2(8 * vox / vy)
        flops += 5.0 * c["n"] * vx * vy * math.log2(max(vx, 2)) * 2
    else:
        # back-projection: 5 flop per voxel and tilt, forward: 10 per ray sample
        cos = np.cos(np.deg2rad(_tilts(c["n"]).astype(np.float64)))
        samples = float(np.sum(np.floor(c["vol_z"] / cos + 1.5))) * vx * vy
        flops += (1 + c["iters"]) * vox * c["n"] * 5 + c["iters"] * samples * 10
    if c.get("patches"):
        flops += 10.0 * c["patches"] * c["n"] * c["nx"] * c["ny"]
    if c.get("bin", 1.0) != 1.0:
        flops += 2.5 * c["n"] * c["nx"] * c["ny"] * math.log2(float(c["nx"]) * c["ny"])
    return nbytes, flops


def work(case):
    c = case
    if c["kind"] in ("slice", "series"):
        b, f = _series_work(c)
    elif c["kind"] == "batch":
        b, f = (sum(v) for v in zip(*(_series_work(m) for m in _members(c))))
    elif c["kind"] == "reproj":
        first, last = find_proj_range(_tilts(c["n"]), c["index"])
        b = 4.0 * c["nx"] * c["ny"] * (last - first + 2)
        f = 5.0 * (last - first + 1) * c["nx"] * c["ny"] * c["vol_z"]
    else:
        m = dict(c, method="wbp", bin=max(20.0 / c["pixel"], 20.0), storage="f32")
        vx, _ = _recon_size(m)
        b, f = _series_work(dict(m, vol_z=int(vx * 0.8) // 2 * 2))
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _cos_sin(tilts):
    a = np.float32(0.017453) * tilts
    return [(float(np.float32(math.cos(float(v)))), float(np.float32(math.sin(float(v))))) for v in a]


def _fill_table(seed, n):
    with np.errstate(over="ignore"):
        x = np.uint64(seed) + np.arange(n, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        x = x ^ (x >> np.uint64(31))
        x = ((x >> np.uint64(32)) * np.uint64(n)) >> np.uint64(32)
    return torch.from_numpy(x.astype(np.int64)).cuda()


def _fill_empty(img, table):
    """Empty pixels take the first non-empty one of their chain, else the mean."""
    flat = img.reshape(-1)
    empty = flat < EMPTY
    if not bool(empty.any()):
        return img
    good = flat[~empty]
    mean = good.mean() if good.numel() else flat.new_zeros(())
    todo = torch.nonzero(empty).reshape(-1)
    nxt, out = table[todo], flat.clone()
    out[todo] = mean
    for _ in range(100):
        ok = ~empty[nxt]
        out[todo[ok]] = flat[nxt[ok]]
        todo, nxt = todo[~ok], nxt[~ok]
        if not todo.numel():
            break
        nxt = table[nxt]
    return out.reshape(img.shape)


def _prestage(c, proj, al):
    ax, ay = _aligned_size(c)
    n, nx, ny = c["n"], c["nx"], c["ny"]
    ang = np.float32(c["axis"]) * (np.float32(3.141592654) / np.float32(180.0))
    ca, sa = math.cos(float(ang)), math.sin(float(ang))
    xc = (torch.arange(ax, device="cuda", dtype=torch.float64) + 0.5 - ax * 0.5)[None, :]
    yc = (torch.arange(ay, device="cuda", dtype=torch.float64) + 0.5 - ay * 0.5)[:, None]
    x0, y0 = xc * ca - yc * sa, xc * sa + yc * ca
    table = _fill_table(al["fill_seed"], ax * ay)
    out = torch.empty((n, ay, ax), device="cuda", dtype=torch.float64)
    for t in range(n):
        xr, yr = x0, y0
        if al["patches"] is not None:
            p = al["patches"][t]
            wx, wy, sw = torch.zeros_like(x0), torch.zeros_like(x0), torch.zeros_like(x0)
            for q in range(p.shape[1]):
                if p[4, q] < np.float32(0.9):
                    continue
                dx, dy = (x0 - float(p[0, q])) / nx, (y0 - float(p[1, q])) / ny
                w = torch.exp(-100.0 * (dx * dx + dy * dy))
                wx += float(p[2, q]) * w
                wy += float(p[3, q]) * w
                sw += w
            ok = sw > 0
            xr = torch.where(ok, x0 + wx / sw, x0)
            yr = torch.where(ok, y0 + wy / sw, y0)
        xr = xr + (float(al["shifts"][t, 0]) + nx * 0.5)
        yr = yr + (float(al["shifts"][t, 1]) + ny * 0.5)
        ix, iy = (xr + 0.5).to(torch.int64), (yr + 0.5).to(torch.int64)
        ok = (ix >= 0) & (ix < nx) & (iy >= 0) & (iy < ny)
        v = proj[t].double()[iy.clamp(0, ny - 1), ix.clamp(0, nx - 1)]
        out[t] = _fill_empty(torch.where(ok, v, SENT), table)
    return out


def _crop(img, bx, by):
    """Fourier crop of the last two axes to by x bx (imaginary parts of the
    DC and Nyquist columns dropped)."""
    ay, ax = img.shape[-2:]
    f = torch.fft.rfft(img, dim=-1)[..., : bx // 2 + 1]
    f = torch.fft.fft(f, dim=-2) / (float(ax) * ay)
    j = torch.arange(by, device=img.device)
    f = f.index_select(-2, torch.where(j <= by // 2, j, j - by + ay))
    f = torch.fft.ifft(f, dim=-2, norm="forward")
    f[..., 0] = f[..., 0].real.to(f.dtype)
    f[..., bx // 2] = f[..., bx // 2].real.to(f.dtype)
    return torch.fft.irfft(f, n=bx, dim=-1, norm="forward")


def _wbp(stack, tilts, vol_z, exclude):
    """Volume [y][z][x], z unflipped, of the aligned stack [n][y][x]."""
    n, ny, px = stack.shape
    p = px // 2 * 2
    cs = _cos_sin(tilts)
    r = torch.arange(p // 2 + 1, device="cuda", dtype=torch.float64) / p
    ramp = 2.0 * r * (0.55 + 0.45 * torch.cos(float(np.float32(6.2831852)) * r)) / p
    w = torch.tensor([v[0] / vol_z for v in cs], device="cuda", dtype=torch.float64)
    sino = torch.fft.rfft(stack[:, :, :p].double() * w[:, None, None], dim=-1) * ramp
    sino = torch.fft.irfft(sino, n=p, dim=-1, norm="forward")
    vx, vz = p, vol_z
    fx = torch.arange(2 * vx, device="cuda", dtype=torch.float64) - vx
    out = torch.empty((ny, vz, vx), device="cuda", dtype=torch.float64)
    step = max(1, min(ny, (1 << 27) // (4 * vx * vz)))
    for y0 in range(0, ny, step):
        rows = sino[:, y0:y0 + step]
        grid = torch.zeros((rows.shape[1], 2 * vz, 2 * vx), device="cuda", dtype=torch.float64)
        cnt = torch.zeros((2 * vz, 2 * vx), device="cuda", dtype=torch.float64)
        fz = (torch.arange(2 * vz, device="cuda", dtype=torch.float64) - vz)[:, None]
        for t in range(n):
            if exclude is not None and exclude[t]:
                continue
            c, s = cs[t]
            u = (fx * c + fz * s) / 2 + p // 2 + 0.5
            ok = ((u >= 0) & (u <= p - 2)).double()
            iu = u.clamp(0, p - 2).to(torch.int64)
            f = (u.clamp(0, p - 2) - iu).reshape(-1)
            i = iu.reshape(-1)
            a, b = rows[t].index_select(1, i), rows[t].index_select(1, i + 1)
            grid += ((a * (1 - f) + b * f) * ok.reshape(-1)).reshape(grid.shape)
            cnt += ok
        grid /= cnt.clamp(min=1)
        out[y0:y0 + step] = _crop(grid, vx, vz)
    return out


def _back(sino, rows, cs, vol, relax, positivity):
    """sino: {tilt: [y][p]}; vol [y][z][x] updated in place."""
    ny, vz, vx = vol.shape
    fx = torch.arange(vx, device="cuda", dtype=torch.float64) - vx * 0.5
    fz = (torch.arange(vz, device="cuda", dtype=torch.float64) - vz * 0.5)[:, None]
    acc = torch.zeros_like(vol)
    cnt = torch.zeros((vz, vx), device="cuda", dtype=torch.float64)
    for t in rows:
        q = sino[t]
        p = q.shape[1]
        u = fx * cs[t][0] + fz * cs[t][1] + p / 2.0
        ok = ((u >= 0) & (u <= p - 2)).double()
        u = u.clamp(0, p - 2)
        i = u.to(torch.int64)
        f = (u - i).reshape(-1)
        i = i.reshape(-1)
        a, b = q.index_select(1, i), q.index_select(1, i + 1)
        acc += ((a * (1 - f) + b * f) * ok.reshape(-1)).reshape(vol.shape)
        cnt += ok
    new = relax * acc / cnt.clamp(min=1) + vol
    if positivity:
        new = new.clamp(min=0)
    vol.copy_(torch.where(cnt > 0, new, vol))


def _forward(vol, c, s, p):
    ny, vz, vx = vol.shape
    length = int(vz / c + 1.5)
    tx = (torch.arange(p, device="cuda", dtype=torch.float64) - 0.5 * p) / c + vx * 0.5
    acc = torch.zeros((ny, p), device="cuda", dtype=torch.float64)
    cnt = torch.zeros(p, device="cuda", dtype=torch.float64)
    for k in range(length):
        fzk = k - length * 0.5
        z = vz * 0.5 + fzk * c
        if z < 0 or z > vz - 2:
            continue
        iz = int(z)
        az = z - iz
        row = vol[:, iz] * (1 - az) + vol[:, iz + 1] * az
        x = tx - fzk * s
        ok = ((x >= 0) & (x <= vx - 2)).double()
        x = x.clamp(0, vx - 2)
        ix = x.to(torch.int64)
        f = x - ix
        acc += (row.index_select(1, ix) * (1 - f) + row.index_select(1, ix + 1) * f) * ok
        cnt += ok
    return torch.where(cnt > 0, acc / cnt.clamp(min=1), SENT)


def _sart(c, stack, al, vol_z):
    n, ny, px = stack.shape
    p = px // 2 * 2
    cs = _cos_sin(al["tilts"])
    raw = [stack[t, :, :p].double() * (cs[t][0] / vol_z) for t in range(n)]
    vol = torch.zeros((ny, vol_z, p), device="cuda", dtype=torch.float64)
    used = [t for t in range(n) if al["exclude"] is None or not al["exclude"][t]]
    _back(raw, used, cs, vol, 1.0, c["positivity"])
    m = c["subsets"]
    if c["interleaved"]:
        subsets = [list(range(s, n, m)) for s in range(m)]
    else:
        subsets = [list(v) for v in np.array_split(np.arange(n), m)]
    relax = float(np.float32(c["relax"])) if c["relax"] > 0 else float(np.float32(1.0) / np.float32(m))
    for _ in range(c["iters"]):
        for sub in subsets:
            diff = {}
            for t in sub:
                fwd = _forward(vol, cs[t][0], cs[t][1], p)
                diff[t] = torch.where(fwd < EMPTY, 0.0, raw[t] - fwd)
            _back(diff, [t for t in sub if t in used], cs, vol, relax, c["positivity"])
    return vol


def _layout(vol, layout):
    if layout == "slice":
        return vol
    if layout == "xzy":
        return vol.flip(1)
    return vol.permute(1, 0, 2)


def _exact_series(c, proj, al):
    stack = _prestage(c, proj, al) if c.get("axis") is not None else proj.double()
    if c.get("bin", 1.0) != 1.0:
        ax, ay = _aligned_size(c)
        bx, by = int(ax / c["bin"]) // 2 * 2, int(ay / c["bin"]) // 2 * 2
        stack = torch.stack([_crop(v, bx, by) for v in stack])
    if c["method"] == "wbp":
        return _wbp(stack, al["tilts"], c["vol_z"], al["exclude"])
    return _sart(c, stack, al, c["vol_z"])


def _seconds(c):
    """About what _exact_series takes."""
    vx, vy = _recon_size(c)
    vox = float(vx) * vy * c["vol_z"]
    if c["method"] == "wbp":
        return c["n"] * vox * 4 / 5e10 + c["n"] * c["nx"] * c["ny"] * c.get("patches", 1) / 1e10
    steps = c["iters"] * c["n"] * c["vol_z"] * 1.4
    return steps * (2e-4 + vx * vy / 2e10) + (1 + c["iters"]) * c["n"] * vox / 5e10


def _exact_reproj(c, proj, tilts):
    first, last = find_proj_range(tilts, c["index"])
    d2r = float(np.float32(0.01745))
    nx, ny, vz = c["nx"], c["ny"], c["vol_z"]
    vx = 2 * nx
    a = float(tilts[c["index"]])
    rad = 4.0 * math.atan(1.0) / 180.0
    fc, fs = float(np.float32(math.cos(rad * a))), float(np.float32(math.sin(rad * a)))
    ray = int(np.float32(np.float32(vz) / np.float32(fc)) + np.float32(0.5))
    need = float(np.float32(0.8) * np.float32(ray))
    fx = (torch.arange(vx, device="cuda", dtype=torch.float64) + 0.5 - vx * 0.5)[None, :]
    fz = (torch.arange(vz, device="cuda", dtype=torch.float64) + 0.5 - vz * 0.5)[:, None]
    out = torch.empty((ny, nx), device="cuda", dtype=torch.float64)
    xp = torch.arange(nx, device="cuda", dtype=torch.float64) + 0.5 - nx * 0.5
    tx = vx * 0.5 + ray * 0.5 * fs + xp / fc
    i = torch.arange(ray, device="cuda", dtype=torch.float64)
    x, z = tx[None, :] - (i * fs)[:, None], (vz * 0.5 - ray * 0.5 * fc + i * fc)[:, None].expand(ray, nx)
    ok = (x >= 0) & (x < vx) & (z >= 0) & (z < vz)
    at = (z.to(torch.int64).clamp(0, vz - 1) * vx + x.to(torch.int64).clamp(0, vx - 1)).reshape(-1)
    for y0 in range(0, ny, 32):
        rows = proj[:, y0:y0 + 32].double()
        num = torch.zeros((rows.shape[1], vz * vx), device="cuda", dtype=torch.float64)
        cnt = torch.zeros((vz, vx), device="cuda", dtype=torch.float64)
        for k in range(first, last + 1):
            v = float(tilts[k]) * d2r
            w = math.cos((a - float(tilts[k])) * d2r)
            u = fx * math.cos(v) + fz * math.sin(v) + nx * 0.5
            inside = ((u >= 0) & (u <= nx - 1)).double()
            iu = u.clamp(0, nx - 1).to(torch.int64).reshape(-1)
            num += rows[k].index_select(1, iu) * (inside.reshape(-1) * math.cos(v) * w)
            cnt += inside * w
        full = (cnt >= 0.001).reshape(-1)
        vol = torch.where(full, num / cnt.reshape(-1).clamp(min=0.001), 0.0)
        hit = (full[at].reshape(ray, nx) & ok).double()
        s = (vol.index_select(1, at).reshape(-1, ray, nx) * hit).sum(1)
        k = hit.sum(0)
        out[y0:y0 + 32] = torch.where(k < need, SENT, s / k.clamp(min=1))
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "reproj":
        proj, al = _inputs(c, seed)
        return _exact_reproj(c, proj, al["tilts"])
    if kind == "thickness":
        return None
    if kind == "batch":
        out = []
        for k, m in enumerate(_members(c)):
            if sum(_seconds(v) for v in _members(c)[: k + 1]) > 18:
                out.append(None)
                continue
            proj, al = _inputs(m, seed + 100 * k)
            out.append(_layout(_exact_series(m, proj, al), "xzy"))
        return out if any(v is not None for v in out) else None
    if _seconds(c) > 18:
        return None
    if kind == "slice":
        proj, al = _inputs(dict(c, ny=32), seed)
        return _exact_series(c, proj[:, 16:17, :].contiguous(), al)[0]
    proj, al = _inputs(c, seed)
    return _layout(_exact_series(c, proj, al), c["layout"])

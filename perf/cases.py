"""The work this framework is measured on: its calls on the sizes a user meets.

Kinds of cases (each one or a few public entry points of mray_amd):
  frame       generate -> prepare -> reconstruct of one image (whole call)
  generate    moments of a volume (f32 or u8), the precomputation of an image
  prepare     Lagrange multipliers of a moment image, dense or compact
  reconstruct the image of given multipliers, dense or compact
  compact     moment counts, index and compact copy of a dense moment image
  train       one optimisation step: image, and its gradients to the voxels
              and to the transfer-function table
  gather      SPH particles sampled onto a grid
  write       prediction coding and entropy coding of a compact image
  read        entropy decoding and coded preparation of a file's section

Inputs are made with torch from the seed alone; exact() evaluates the same
discretisation (the reference's float sample positions and phases) in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from mray_amd import autograd as ag
from mray_amd import hip, synth
from mray_amd import tf as tfmod
from mray_amd.types import GenParams, RecParams

DEV = "cuda"
PI = math.pi
# word widths of the entropy-coded moments: what the quantisation-curve search
# picks for a 50-moment frame at 10 bits, its last width for further moments
CURVE = [16, 10, 9, 8, 8] + [7] * 9 + [6] * 28 + [5] * 3 + [4, 3]


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # the smallest frames (previews, unit-sized images): launches and latency
        dict(name="frame_64x48_m30", kind="frame", vol="signal", n=48, W=64, H=48, m=30, cam="ortho"),
        # an ordinary frame, odd sizes: the analytic-signal configuration's
        # 128^3 grid and 30 moments, generate -> prepare -> reconstruct
        dict(name="frame_509x387_m30", kind="frame", vol="signal", n=128, W=509, H=387, m=30, cam="ortho"),
        # the precision study's three stages, each by itself: 1024^3 f32
        # mixing layer, perspective 1024 x 1024 rays, 50 moments
        dict(name="generate_f32_1024_m50", kind="generate", vol="layer", n=1024, W=1024, H=1024, m=50, cam="persp"),
        dict(name="prepare_1024_m50", kind="prepare", W=1024, H=1024, m=50, compact=False, wide=True),
        dict(name="reconstruct_1024_m50", kind="reconstruct", W=1024, H=1024, m=50, steps=1150, compact=False,
             wide=True),
        # the large volume: 2048 x 2048 x 1920 u8, 2048 x 2048 rays, 100 moments
        dict(name="generate_u8_2048_m100", kind="generate", vol="blobs", n=2048, W=2048, H=2048, m=100, cam="persp"),
        # the compaction of such an image (a quarter of its pixels)
        dict(name="compact_1024_m100", kind="compact", W=1024, H=1021, m=100),
        # the compact image prepared (ragged counts)
        dict(name="prepare_compact_1000_m96", kind="prepare", W=1000, H=777, m=96, compact=True, wide=True),
        # volume and transfer-function fitting: 256^3 f32, 512 x 512 rays, 40 moments
        dict(name="train_512_m40", kind="train", vol="signal", n=256, W=512, H=512, m=40, cam="ortho"),
        # 20 M particles gathered onto 512 x 512 x 256 voxels
        dict(name="gather_20M_512", kind="gather", particles=20_000_000, n=512, h=0.004),
        # the eval's file options: prediction-coded, entropy-coded moments
        dict(name="write_640_m50", kind="write", W=640, H=641, m=50),
        dict(name="read_640_m50", kind="read", W=640, H=641, m=50),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "generate", "generate", "prepare", "prepare", "reconstruct", "reconstruct", "compact",
                       "train", "gather", "write", "read"])
    W, H = _log(rng, 40, 1024), _log(rng, 40, 1024)
    cam = rng.choice(["ortho", "persp"])
    if kind == "frame":
        return dict(kind=kind, vol=rng.choice(["signal", "layer"]), n=_log(rng, 32, 512), W=W, H=H,
                    m=rng.randint(4, 60), cam=cam)
    if kind == "generate":
        return dict(kind=kind, vol=rng.choice(["signal", "layer", "blobs"]), n=_log(rng, 48, 1024), W=W, H=H,
                    m=rng.randint(4, 128), cam=cam)
    if kind == "prepare":
        return dict(kind=kind, W=W, H=H, m=rng.randint(4, 128), compact=rng.random() < 0.5, wide=rng.random() < 0.5)
    if kind == "reconstruct":
        return dict(kind=kind, W=W, H=H, m=rng.randint(4, 128), steps=_log(rng, 100, 2000),
                    compact=rng.random() < 0.5, wide=rng.random() < 0.5)
    if kind == "compact":
        return dict(kind=kind, W=W, H=H, m=rng.randint(8, 100))
    if kind == "train":
        return dict(kind=kind, vol=rng.choice(["signal", "layer"]), n=_log(rng, 32, 256), W=_log(rng, 40, 512),
                    H=_log(rng, 40, 512), m=rng.randint(8, 64), cam=cam)
    if kind == "gather":
        return dict(kind=kind, particles=_log(rng, 20_000, 10_000_000), n=_log(rng, 64, 512),
                    h=rng.choice([0.004, 0.006, 0.01]))
    return dict(kind=kind, W=_log(rng, 40, 600), H=_log(rng, 40, 600), m=rng.randint(8, 64))


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _axis(n, cells):
    """Lower lattice index and smooth weight of n positions i / n over `cells` lattice cells."""
    p = torch.arange(n, device=DEV, dtype=torch.float32) * (cells / n)
    i = p.floor().clamp(max=cells - 1)
    f = p - i
    return i.long(), f * f * (3 - 2 * f)


def _noise_planes(lattices, z, nz, ny, nx):
    """Value noise in [-1, 1] of the z planes `z` (a slice) from lattices of doubling resolution."""
    total, norm = 0.0, 0.0
    for o, lat in enumerate(lattices):
        c = lat.shape[0] - 1
        i, f = _axis(nz, c)
        i, f = i[z], f[z][:, None, None]
        a = lat[i] * (1 - f) + lat[i + 1] * f
        i, f = _axis(ny, c)
        a = a[:, i] * (1 - f)[None, :, None] + a[:, i + 1] * f[None, :, None]
        i, f = _axis(nx, c)
        a = a[:, :, i] * (1 - f) + a[:, :, i + 1] * f
        total = total + a * 0.5 ** o
        norm += 0.5 ** o
    return total / norm


def _lattices(g, base, octaves):
    return [2 * torch.rand((base * 2 ** o + 1,) * 3, device=DEV, generator=g) - 1 for o in range(octaves)]


def _volume(kind, n, seed):
    """(voxels, dmin, dmax): the analytic signal on [-1,1]^3 or a mixing layer
    on [0,1]^3 (f32), or noise and blobs in a 2048:2048:1920 box (u8)."""
    g = _gen(seed)
    u = torch.rand(64, device=DEV, generator=g)
    if kind == "signal":
        c = torch.arange(n, device=DEV, dtype=torch.float32) * (2.0 / n) - 1.0
        fm, a, cx, cy, sz = 5.0 + 2.0 * float(u[0]), 0.25, 0.2 * float(u[1]), 0.2 * float(u[2]), float(u[3])
        r = torch.sqrt((c[None, :] - cx) ** 2 + (c[:, None] - cy) ** 2)
        rho = torch.cos(2 * PI * fm * torch.cos(PI * r / 2))
        v = (1 - torch.sin(PI * (c + 0.1 * sz) / 2)[:, None, None] + a * (1 + rho)[None]) / (2 * (1 + a))
        return v.contiguous(), (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
    if kind == "layer":
        lat = _lattices(g, 8, 4)
        c = torch.arange(n, device=DEV, dtype=torch.float32) / n
        h = torch.zeros((n, n), device=DEV)
        for k in range(16):
            th, ph, amp = 2 * PI * float(u[k]), 2 * PI * float(u[16 + k]), 0.02 / (k + 1) * (2 * float(u[32 + k]) - 1)
            h += amp * torch.sin(2 * PI * (k + 1) * (c[None, :] * math.cos(th) + c[:, None] * math.sin(th)) + ph)
        v = torch.empty((n, n, n), device=DEV)
        for z in range(0, n, 32):
            s = slice(z, min(n, z + 32))
            v[s] = 0.5 + 0.5 * torch.tanh((c[s, None, None] - 0.5 - h) / 0.01) + 0.05 * _noise_planes(lat, s, n, n, n)
        return v, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0)
    nz = max(2, n * 1920 // 2048)
    lat = _lattices(g, 4, 6)
    b = torch.rand((64, 5), device=DEV, generator=g)
    ext = (1.0, 1.0, nz / n)
    sig = ((20 + 60 * b[:, 3]) / 2048)[:, None]
    gx, gy, gz = (torch.exp(-0.5 * ((torch.arange(k, device=DEV) / n)[None] - (b[:, d] * ext[d])[:, None]) ** 2 / sig ** 2)
                  for d, k in enumerate((n, n, nz)))
    gx = gx * (0.4 + 0.6 * b[:, 4])[:, None]
    v = torch.empty((nz, n, n), device=DEV, dtype=torch.uint8)
    for z in range(0, nz, 16):
        s = slice(z, min(nz, z + 16))
        t = ((0.5 + 0.5 * _noise_planes(lat, s, nz, n, n) - 0.3) / 0.4).clamp(0, 1)
        blobs = (gz[:, s].t()[:, None, :] * gy.t()[None]).reshape(-1, 64) @ gx
        v[s] = (255 * (0.5 * t * t * (3 - 2 * t) + blobs.view(t.shape)).clamp(0, 1) + 0.5).to(torch.uint8)
    return v, (0.0, 0.0, 0.0), ext


def _camera(case, dmin, dmax):
    if case["cam"] == "ortho":
        return synth.ortho_camera(pos=tuple((a + b) / 2 for a, b in zip(dmin[:2], dmax[:2])) + (dmin[2] - 2.0,))
    size = dmax[0] - dmin[0]
    pos = ((dmin[0] + dmax[0]) / 2, (dmin[1] + dmax[1]) / 2, dmin[2] - size)
    return synth.perspective_camera(position=pos, fov_half_deg=25.0, znear=0.01, aspect=case["W"] / case["H"])


def _scene(case, seed):
    vox, dmin, dmax = _volume(case["vol"], case["n"], seed)
    # half a voxel per step, one voxel for the large u8 volumes
    step = (1.0 if case["vol"] == "blobs" else 0.5) * (dmax[0] - dmin[0]) / case["n"]
    gp = GenParams(step_size=step, transform_to_bounds=1, transform_bound_eps=0.01, compact_image=0,
                   prediction_coding=0, bias=1e-4)
    rp = RecParams(step_size=step, bias=1e-3, early_ray_termination=0.99, medium_emission=1.0)
    table = torch.from_numpy(tfmod.table_from_rgba8(synth.tf_ramps(int(seed) % 1000), step * 16.0)).to(DEV)
    return vox, dmin, dmax, _camera(case, dmin, dmax), gp, rp, table


def _field(g, W, H, count, cells=12):
    """`count` smooth fields over the image with values in (0, 1): (H*W, count)."""
    low = torch.rand((1, count, cells, cells), device=DEV, generator=g)
    return F.interpolate(low, size=(H, W), mode="bilinear", align_corners=True)[0].reshape(count, -1).t().contiguous()


def _moment_field(case, seed):
    """Moments (H*W, m) of smooth piecewise-constant densities along the rays
    (up to six materials, interfaces blurred by 0.5 to 5 % of a ray), f32, and
    packed bounds; the image's corners are rays that miss the volume."""
    W, H, m = case["W"], case["H"], case["m"]
    g = _gen(seed)
    cuts = torch.cumsum(0.1 + _field(g, W, H, 6), 1).double()
    phi = torch.cat([torch.zeros_like(cuts[:, :1]), cuts], 1) / cuts[:, -1:] * PI - PI
    val = (0.02 + 0.96 * _field(g, W, H, 6)).double()
    blur = (0.005 + 0.045 * _field(g, W, H, 1)[:, 0]).double() * PI
    out = torch.empty((W * H, m), device=DEV)
    out[:, 0] = ((phi[:, 1:] - phi[:, :-1]) * val).sum(1) / PI
    for j in range(1, m):
        sn = torch.sin(j * phi)
        out[:, j] = ((sn[:, 1:] - sn[:, :-1]) * val).sum(1) / (PI * j) * torch.exp(-0.5 * (j * blur) ** 2)
    lo, hi = _field(g, W, H, 2).t()
    bounds = (0.2 * lo * 65535).int() | ((0.7 + 0.3 * hi) * 65535).int() << 16
    y, x = torch.meshgrid(torch.linspace(-1, 1, H, device=DEV), torch.linspace(-1, 1, W, device=DEV), indexing="ij")
    miss = (x * x + y * y > 1.85).reshape(-1)
    out[miss] = 0
    bounds[miss] = 0
    return out.contiguous(), bounds.contiguous(), miss


def _compacted(case, seed):
    """(compact moments, index, bounds): each pixel's first 8 to m moments (the
    same counts for every seed, so that all have one size), none of rays that miss."""
    W, H, m = case["W"], case["H"], case["m"]
    mo, bounds, miss = _moment_field(case, seed)
    lo = min(8, m)
    counts = (lo + (m + 1 - lo) * _field(_gen(m), W, H, 1)[:, 0]).int().clamp(max=m)
    counts[miss] = 0
    index = torch.zeros(W * H + 1, device=DEV, dtype=torch.int32)
    index[1:] = torch.cumsum(counts, 0)
    data = mo[torch.arange(m, device=DEV)[None] < counts[:, None]]
    return data.contiguous(), index, bounds


def _dense(values, index, m, dtype=torch.float64):
    """Compact values laid out densely, zero past each pixel's count."""
    counts = (index[1:] - index[:-1]).long()
    out = torch.zeros((counts.numel(), m), device=DEV, dtype=dtype)
    out[torch.arange(m, device=DEV)[None] < counts[:, None]] = values.to(dtype)
    return out


def _march(case):
    """Camera, box, parameters and table of a reconstruct call of case["steps"] steps through the box."""
    dmin, dmax = (0.0, 0.0, 0.0), (1.0, 1.0, 1.0)
    step = 1.0 / case["steps"]
    cam = _camera(dict(case, cam="persp"), dmin, dmax)
    rp = RecParams(step_size=step, bias=1e-3, early_ray_termination=0.99, medium_emission=1.0)
    table = torch.from_numpy(tfmod.table_from_rgba8(synth.tf_ramps(case["m"]), step * 16.0)).to(DEV)
    return cam, dmin, dmax, rp, table


def _particles(case, seed):
    """Particles of a mixture of 32 anisotropic Gaussians in [0,1] x [0,1] x [0,0.5], varying values."""
    n, g = case["particles"], _gen(seed)
    box = torch.tensor([1.0, 1.0, 0.5], device=DEV)
    centre = (0.15 + 0.7 * torch.rand((32, 3), device=DEV, generator=g)) * box
    sigma = (0.01 + 0.06 * torch.rand((32, 3), device=DEV, generator=g)) * box
    comp = torch.randint(0, 32, (n,), device=DEV, generator=g)
    p = centre[comp] + sigma[comp] * torch.randn((n, 3), device=DEV, generator=g)
    p = torch.minimum(p.clamp(min=0.0), box * (1 - 1e-6))
    v = 0.5 + torch.rand(n, device=DEV, generator=g)
    return [p[:, 0].contiguous(), p[:, 1].contiguous(), p[:, 2].contiguous(), v]


def _widths(m):
    return (CURVE + [CURVE[-1]] * m)[:m]


def prepare(case, seed):
    hip.init(0)
    k = case["kind"]
    s = dict(case=case)
    if k in ("frame", "generate", "train"):
        vox, dmin, dmax, cam, gp, rp, table = _scene(case, seed)
        s.update(vox=vox, dmin=dmin, dmax=dmax, cam=cam, gp=gp, rp=rp, table=table)
        if k == "train":
            g = _gen(seed + 3)
            s["target"] = torch.rand((case["H"], case["W"], 4), device=DEV, generator=g)
        else:
            s["volume"] = hip.Volume(vox, dmin, dmax)
    elif k in ("prepare", "reconstruct"):
        if case["compact"]:
            s["moments"], s["index"], s["bounds"] = _compacted(case, seed)
        else:
            s["moments"], s["bounds"], _ = _moment_field(case, seed)
            s["index"] = None
        if k == "reconstruct":
            cam, dmin, dmax, rp, table = _march(case)
            mo = s["moments"] if s["index"] is None else _dense(s["moments"], s["index"], case["m"], torch.float32)
            lag = _in_chunks(lambda a, n: _multipliers(a, rp.bias, n), mo, _counts(s, case["m"]), case["m"])
            if s["index"] is not None:
                lag = lag[torch.arange(case["m"], device=DEV)[None] < _counts(s, case["m"])[:, None]]
            lag = lag.contiguous()
            s.update(cam=cam, dmin=dmin, dmax=dmax, rp=rp, table=table,
                     lagrange=lag if case["wide"] else lag.float())
    elif k == "compact":
        s["moments"], s["bounds"], _ = _moment_field(case, seed)
        # compact images differ in size: each is kept in a buffer of the dense one's
        s["kept"] = torch.zeros(s["moments"].numel(), device=DEV)
    elif k == "gather":
        s["parts"] = _particles(case, seed)
    else:
        s["data"], s["index"], s["bounds"] = _compacted(case, seed)
        if k == "read":
            data = s["data"].clone()
            W, H, m = case["W"], case["H"], case["m"]
            s["params"] = hip.prediction_encode(data, s["index"], W, H, m, 0, 1e-4)
            s["section"] = hip.entropy_encode(data, s["index"], W, H, m, True, _widths(m))
            del s["data"]
        else:  # sections differ in size: each is kept in a buffer of two bytes a moment, as a file's writer would
            s["kept"] = np.zeros(2 * s["data"].numel() + 65536, np.uint8)
    return s


def _keep(buf, values):
    """`values` at the start of a buffer, zeros behind them."""
    n = values.shape[0]
    buf[:n] = values
    buf[n:] = 0
    return buf


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "gather":
        n = case["n"]
        x, y, z, v = s["parts"]
        return hip.particles_to_grid(x, y, z, v, case["h"], (0.0, 0.0, 0.0), (1.0, 1.0, 0.5), n, n, n // 2)
    W, H, m = case["W"], case["H"], case["m"]
    if k == "generate":
        mo, b, _ = hip.generate(s["volume"], s["cam"], s["gp"], W, H, m)
        return mo, b
    if k == "frame":
        mo, b, _ = hip.generate(s["volume"], s["cam"], s["gp"], W, H, m)
        lag = hip.prepare(mo, W, H, m, s["rp"].bias, form="mixed64")
        rgba, _ = hip.reconstruct(s["cam"], s["dmin"], s["dmax"], lag, W, H, m, s["table"], s["rp"], bounds=b)
        return mo, b, rgba
    if k == "train":
        vox, table = s["vox"].detach().requires_grad_(), s["table"].detach().requires_grad_()
        rgba = ag.render(vox, s["dmin"], s["dmax"], s["cam"], s["gp"], W, H, m, table, s["rp"])
        loss = ((rgba - s["target"]) ** 2).mean()
        g_vox, g_table = torch.autograd.grad(loss, (vox, table))
        return rgba.detach(), g_vox, g_table
    if k == "prepare":
        return hip.prepare(s["moments"], W, H, m, 1e-3, form="mixed64" if case["wide"] else "mixed", index=s["index"])
    if k == "reconstruct":
        rgba, _ = hip.reconstruct(s["cam"], s["dmin"], s["dmax"], s["lagrange"], W, H, m, s["table"], s["rp"],
                                  index=s["index"], bounds=s["bounds"])
        return rgba
    if k == "compact":
        data, index = hip.compact_image(s["moments"], W, H, m, 1e-3, bounds=s["bounds"], count_range=(8, m))
        return _keep(s["kept"], data), index
    if k == "write":
        data = s["data"].clone()
        params = hip.prediction_encode(data, s["index"], W, H, m, 0, 1e-4)
        section = hip.entropy_encode(data, s["index"], W, H, m, True, _widths(m))
        return _keep(s["kept"], section), section.size, params
    coded = hip.entropy_decode(s["section"], s["index"], W, H, m, True, _widths(m))
    return hip.prepare_coded(coded, W, H, m, 0, s["params"], index=s["index"])


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _samples(case):
    """Samples of a frame: the box's path lengths of a coarse grid of its rays over the step."""
    nz = case["n"] * (1920 / 2048 if case["vol"] == "blobs" else 1)
    per = (1 if case["vol"] == "blobs" else 2)
    if case["cam"] == "ortho":
        return case["W"] * case["H"] * nz * per
    a, t = case["W"] / case["H"], math.tan(math.radians(25))
    x, y = np.meshgrid(np.linspace(-t * a, t * a, 64), np.linspace(-t, t, 64))
    out = np.minimum(1 + nz / case["n"], 0.5 / np.maximum(np.maximum(abs(x), abs(y)), 1e-9))
    return case["W"] * case["H"] * case["n"] * per * float((np.maximum(out - 1, 0) * np.sqrt(1 + x * x + y * y)).mean())


def work(case):
    k, m = case["kind"], case.get("m", 0)
    if k == "gather":
        n = case["n"]
        out = n * n * (n // 2)
        # each particle touches the voxels within h of it
        touched = case["particles"] * 4.19 * (case["h"] * n) ** 3
        return {"bytes": 16.0 * case["particles"] + 4.0 * out, "flops": 20.0 * touched}
    rays = case["W"] * case["H"]
    if k in ("frame", "generate", "train"):
        ns = _samples(case)
        vol = case["n"] ** 3 * (1920 / 2048 if case["vol"] == "blobs" else 4.0)
        # a cosine and a multiply-add per moment and sample, the sample itself
        w = {"bytes": vol + rays * (4.0 * m + 4), "flops": ns * (4.0 * m + 30)}
        if k == "generate":
            return w
        back = 3.0 if k == "train" else 1.0  # forward, and twice that backward
        return {"bytes": w["bytes"] + rays * (12.0 * m + 20) * back + (2 * vol if k == "train" else 0),
                "flops": (w["flops"] + rays * 16.0 * m * m + ns * (4.0 * m + 48)) * back}
    mean = (8 + m) / 2 if case.get("compact") or k in ("write", "read") else m
    if k == "prepare":
        return {"bytes": rays * mean * (12.0 if case["wide"] else 8.0), "flops": rays * 16.0 * mean * mean}
    if k == "reconstruct":
        return {"bytes": rays * (mean * (8.0 if case["wide"] else 4.0) + 20),
                "flops": rays * case["steps"] * (4.0 * mean + 48)}
    if k == "compact":  # a Levinson solve and an extension of the moments per step of a binary search
        return {"bytes": rays * 8.0 * m, "flops": rays * 16.0 * m * m * max(1.0, math.log2(m))}
    # a symbol per moment beside the solve per pixel of the prediction (or its inverse) and the preparation
    return {"bytes": rays * mean * 5.0, "flops": rays * mean * (16.0 * mean + 40)}


def tolerance(case):
    """About four times the distance from exact() that was measured: moments
    and f32 multipliers are rounded to f32 once, FP64 multipliers depend on
    the order of the sums through the conditioning of the Toeplitz system, a
    ray's early termination can flip by one step, and a frame's image and the
    gradients pass the bounded MESE, which amplifies the rounding of its f32
    moments."""
    k = case["kind"]
    if k in ("compact", "write", "read"):
        return "exact"  # counts, codes and decoded values are the reference's FP32 arithmetic bit for bit
    if k == "generate":
        return {"rel": 2e-7, "max": 4e-6}
    if k == "gather":
        return {"rel": 1e-6, "max": 1e-4}
    if k == "prepare":
        return {"rel": 1e-8, "max": 1e-6} if case["wide"] else {"rel": 2.5e-7, "max": 4e-6}
    if k == "reconstruct":
        return {"rel": 2e-5, "max": 0.05}
    if k == "frame":
        return {"rel": 2e-3, "max": 0.4}
    return {"rel": 1e-2, "max": 0.5}


# --------------------------------------------------------------------------
# 64 bits
# --------------------------------------------------------------------------
def _f32div(a, b):
    """The IEEE single-precision quotient (through FP64: the double rounding is harmless)."""
    b = b if torch.is_tensor(b) else torch.tensor(float(np.float32(b)), device=DEV, dtype=torch.float64)
    return (a.double() / b.double()).float()


def _f(x):
    return float(np.float32(x))


def _rays(cam, dmin, dmax, W, H):
    """Float ray origins, directions and slab interval of every pixel, as the reference forms them."""
    y, x = torch.meshgrid(torch.arange(H, device=DEV), torch.arange(W, device=DEV), indexing="ij")
    nx = _f32div(x.reshape(-1).float(), W) * 2.0 - 1.0
    ny = _f32div(y.reshape(-1).float(), H) * 2.0 - 1.0
    if cam["orthographic"]:
        o = [(_f(cam["position"][i]) + nx * _f(cam["right"][i])) + ny * _f(cam["up"][i]) for i in range(3)]
        d = [torch.full_like(nx, _f(cam["dir"][i])) for i in range(3)]
    else:
        o = [torch.full_like(nx, _f(cam["position"][i])) for i in range(3)]
        px, py = nx * _f(cam["aspect"]) * _f(cam["scale"]), ny * _f(cam["scale"])
        M = [_f(v) for v in cam["transform"]]
        v = [px * M[4 * r] + py * M[4 * r + 1] + M[4 * r + 2] * -1.0 + M[4 * r + 3] * 0.0 for r in range(3)]
        n2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2]
        inv = _f32div(torch.ones_like(n2), n2.double().sqrt().float())
        d = [c * inv for c in v]
    near = far = None
    for i in range(3):
        r = _f32div(torch.ones_like(d[i]), d[i])
        a, b = r * (_f(dmin[i]) - o[i]), r * (_f(dmax[i]) - o[i])
        lo, hi = torch.where(b < a, b, a), torch.where(b > a, b, a)
        near = lo if near is None else torch.where(near > lo, near, lo)
        far = hi if far is None else torch.where(far < hi, far, hi)
    hit = far > near
    near = torch.where(near > _f(cam["znear"]), near, torch.full_like(near, _f(cam["znear"])))
    return o, d, near, far, hit & (far > 0)


def _corners(vox, dmin, dmax, p):
    """Trilinear corner indices and float weights of positions p (three float tensors)."""
    n = [vox.shape[2], vox.shape[1], vox.shape[0]]
    lo, hi, w = [], [], []
    for i in range(3):
        ip = _f32div(p[i] - _f(dmin[i]), float(np.float32(dmax[i]) - np.float32(dmin[i]))) * float(n[i])
        fl = ip.floor()
        w.append(ip - fl)
        lo.append(fl.long().clamp(0, n[i] - 1))
        hi.append((fl.long() + 1).clamp(0, n[i] - 1))
    at, wt = [], []
    for z, y, x in ((0, 0, 0), (0, 0, 1), (0, 1, 0), (0, 1, 1), (1, 0, 0), (1, 0, 1), (1, 1, 0), (1, 1, 1)):
        at.append(((hi if z else lo)[2] * n[1] + (hi if y else lo)[1]) * n[0] + (hi if x else lo)[0])
        wt.append((w[0] if x else 1.0 - w[0]) * (w[1] if y else 1.0 - w[1]) * (w[2] if z else 1.0 - w[2]))
    return at, wt


def _density(vox, at, wt):
    flat = vox.reshape(-1)
    acc = None
    for a, w in zip(at, wt):
        v = flat[a].float()
        v = _f32div(v, 255.0) if vox.dtype == torch.uint8 else v
        acc = w * v if acc is None else acc + w * v
    return acc.clamp(0.0, 1.0)


class _Segments:
    """The samples and phase segments of a group of rays that hit the box, (K, R) tensors."""

    def __init__(self, vox, dmin, dmax, gp, o, d, near, far, keep_corners=False):
        s = torch.tensor(_f(gp.step_size), device=DEV)
        rng = far - near
        pti = (PI / rng.double()).float()
        dphi = (PI * _f32div(s.expand_as(rng), rng).double()).float()
        ts, t = [near], near
        while True:
            go = t + s < far
            if not bool(go.any()):
                break
            t = torch.where(go, t + s, t)
            ts.append(t)
        ts.append(far)
        t = torch.stack(ts)
        K = t.shape[0]
        # a ray's march stops at its last t < far: later rows repeat it (no segment), the last row is far
        self.live = torch.cat([t[1:-1] > t[:-2], torch.ones_like(t[:1], dtype=torch.bool)])
        ph = ((t - near) * pti).double() - PI
        ph = ph.float()
        ph[0] = _f(-PI)
        self.p = ph[1:].double()
        self.p[-1] = 0.0
        seg = torch.empty((K - 1, near.numel()), device=DEV)
        seg[:-1] = dphi
        seg[-1] = 0.0 - ph[-2]
        self.seg = seg.double()
        self.u = (self.p.float() - seg).double()
        f, self.at, self.wt = [], [], []
        for k in range(0, K, 64):
            tk = t[k:k + 64]
            at, wt = _corners(vox, dmin, dmax, [o[i] + tk * d[i] for i in range(3)])
            f.append(_density(vox, at, wt))
            if keep_corners:
                self.at.append(torch.stack(at))
                self.wt.append(torch.stack(wt))
        f = torch.cat(f)
        self.lo, self.hi = f.min(0).values.clamp(max=1.0), f.max(0).values.clamp(min=0.0)
        if gp.transform_to_bounds:
            e = _f(gp.transform_bound_eps)
            self.lo, self.hi = (self.lo - e).clamp(min=0.0), (self.hi + e).clamp(max=1.0)
        self.f = f.double()
        self.inv = 1.0 / (self.hi.double() - self.lo.double())

    def terms(self, j):
        """The linear terms of moment j in (slope, end value, start value) per segment, zero where there is none."""
        return ((torch.cos(j * self.p) - torch.cos(j * self.u)) / (j * j) * self.live,
                torch.sin(j * self.p) / j * self.live, torch.sin(j * self.u) / j * self.live)

    def moments(self, m):
        sg = (self.p - self.u)
        f0, f1 = self.f[:-1], self.f[1:]
        g = (f1 - f0) / self.seg
        fe = f0 + g * sg
        out = torch.empty((f0.shape[1], m), device=DEV, dtype=torch.float64)
        out[:, 0] = ((sg * (f0 + 0.5 * g * sg) * self.live).sum(0) / PI - self.lo.double()) * self.inv
        for j in range(1, m):
            a, b, c = self.terms(j)
            out[:, j] = (g * a + fe * b - f0 * c).sum(0) / PI * self.inv
        return out

    def moments_adjoint(self, gm):
        """dL/df (K, R) of dL/dmoments (R, m)."""
        sg = (self.p - self.u)
        gm = gm.double() * self.inv[:, None] / PI
        gf = torch.zeros_like(self.f)
        w = gm[:, 0] * self.live * sg
        ga, ge, g0 = 0.5 * sg * w, torch.zeros_like(w), w.clone()
        for j in range(1, gm.shape[1]):
            a, b, c = self.terms(j)
            ga += gm[:, j] * a
            ge += gm[:, j] * b
            g0 -= gm[:, j] * c
        ga += ge * sg
        g0 += ge
        gf[1:] += ga / self.seg
        gf[:-1] += g0 - ga / self.seg
        return gf


def _multipliers(mo, bias, counts):
    """Bounded-MESE multipliers (R, m) of moments (R, m) in FP64; entries from a pixel's count on are zero."""
    bias = _f(bias)
    m = mo.shape[1]
    t = (1.0 - bias) * mo.double()
    t = torch.cat([t[:, :1] + 0.5 * bias, t[:, 1:]], 1)
    keep = (torch.arange(m, device=mo.device)[None] < counts[:, None])
    t = torch.where(keep, t, torch.zeros_like(t))
    phase = PI * t[:, 0] - 0.5 * PI
    e0 = torch.complex(torch.cos(phase), torch.sin(phase)) / (4 * PI)
    jt = t * torch.arange(m, device=mo.device)
    E = e0[:, None]
    for l in range(1, m):
        E = torch.cat([E, (2j * PI / l) * (jt[:, 1:l + 1].flip(1) * E).sum(1, keepdim=True)], 1)
    E = torch.where(keep, E, torch.zeros_like(E))
    E2 = torch.cat([2 * E[:, :1], E[:, 1:]], 1)
    A = torch.complex(1.0 / E2[:, :1].real, torch.zeros_like(E2[:, :1].real))
    valid = torch.ones_like(A[:, :1].real)
    for j in range(1, m):
        u = (A * E2[:, 1:j + 1].flip(1)).sum(1, keepdim=True) * valid
        ok = ((u.real ** 2 + u.imag ** 2) < 1.0).double()
        valid = valid * ok * keep[:, j:j + 1]
        u = u * valid
        fac = 1.0 / (1.0 - (u.real ** 2 + u.imag ** 2))
        z = torch.zeros_like(A[:, :1])
        A = fac * (torch.cat([A, z], 1) - torch.cat([z, A.flip(1).conj()], 1) * u)
    P = 2 * PI * A
    R = torch.stack([(P[:, :m - k] * P[:, k:].conj()).sum(1) for k in range(m)], 1)
    lam = torch.stack([(R[:, k:] * E[:, :m - k]).sum(1).imag for k in range(m)], 1)
    return lam / (PI * P[:, :1].real) * keep


def _in_chunks(fn, a, counts, m):
    rows = max(256, (1 << 22) // m)
    return torch.cat([fn(a[i:i + rows], counts[i:i + rows]) for i in range(0, a.shape[0], rows)])


def _counts(s, m):
    if s.get("index") is None:
        return torch.full((s["moments"].shape[0],), m, device=DEV, dtype=torch.int64)
    return (s["index"][1:] - s["index"][:-1]).long()


def _atan(t):
    """The reference's arctangent polynomial (float coefficients) in FP64."""
    a = t.abs()
    big = a > 1.0
    x = torch.where(big, 1.0 / torch.where(big, a, torch.ones_like(a)), a)
    y = x * x
    z = y * _f(0.020835) - _f(0.085133)
    z = y * z + _f(0.180141)
    z = y * z - _f(0.330299)
    q = y * z + _f(0.999866)
    r = x * q + torch.where(big, q * x * -2.0 + _f(1.570796), torch.zeros_like(a))
    return torch.where(t < 0, -r, r)


def _image(lam, lo, hi, near, far, table, rp):
    """RGBA (R, 4) of rays that hit, from multipliers (R, m) and density bounds, differentiable in lam and table."""
    step = torch.tensor(_f(rp.step_size), device=DEV)
    rng = far - near
    dp = (PI * _f32div(step.expand_as(rng), rng).double()).float()
    t, p = near, torch.full_like(near, _f(-PI))
    ps, lives = [p], []
    while True:
        go = t <= far
        if not bool(go.any()):
            break
        t, p = t + step, p + dp
        ps.append(p)
        lives.append(go)
    ph = torch.stack(ps).double().clamp(-PI, 0.0)
    live = torch.stack(lives)
    S = lam[:, 0].expand(ph.shape)
    for l in range(1, lam.shape[1]):
        S = S + 2 * lam[:, l] * torch.cos(l * ph)
    rho = (_atan(S) / PI + 0.5) * (hi - lo) + lo
    fs, bs = rho[:-1] * 256.0, rho[1:] * 256.0
    ay = bs - bs.detach().floor()
    xl = fs.detach().floor().long()
    w1 = (ay * live)[..., None]
    w0 = ((1 - ay) * live)[..., None]
    c = w0 * table[xl.clamp(0, 255)] + w1 * table[(xl + 1).clamp(0, 255)]
    tau = torch.cumsum(c[..., 3], 0)
    T = torch.exp(-tau)
    end = (1 - T.detach() >= _f(rp.early_ray_termination))
    before = torch.cat([torch.ones_like(T[:1]), T[:-1]])
    on = (torch.cumsum(end.int(), 0) - end.int()) == 0  # the step that terminates still emits
    rgb = (_f(rp.medium_emission) * c[..., :3] * (before * on)[..., None]).sum(0)
    alpha = torch.where(end.any(0), torch.ones_like(T[0]), 1 - T[-1])
    return torch.cat([rgb, alpha[:, None]], 1)


def _quantised(lo, hi):
    """The 16-bit bounds a frame keeps, as densities."""
    return (lo * 65535.0).int().double() / 65535.0, (hi * 65535.0).int().double() / 65535.0


def exact(case, seed):
    k = case["kind"]
    if k in ("compact", "write", "read"):
        return None  # decisions, codes and values defined by the reference's FP32 arithmetic
    s = prepare(case, seed)
    if k == "gather":
        return _gather64(s) if case["particles"] * (case["h"] * case["n"] + 1) ** 3 < 1.5e8 else None
    W, H, m = case["W"], case["H"], case["m"]
    if k == "prepare":
        mo = s["moments"] if s["index"] is None else _dense(s["moments"], s["index"], m, torch.float32)
        lam = _in_chunks(lambda a, n: _multipliers(a, 1e-3, n), mo, _counts(s, m), m)
        return lam if s["index"] is None else lam[torch.arange(m, device=DEV)[None] < _counts(s, m)[:, None]]
    if k == "reconstruct":
        if W * H * case["steps"] * m > 8e10:
            return None
        lam = s["lagrange"].double() if s["index"] is None else _dense(s["lagrange"], s["index"], m)
        b = s["bounds"].long()
        lo, hi = (b & 65535).double() / 65535.0, ((b >> 16) & 65535).double() / 65535.0
        _, _, near, far, hit = _rays(s["cam"], s["dmin"], s["dmax"], W, H)
        out = torch.zeros((W * H, 4), device=DEV, dtype=torch.float64)
        for r in torch.nonzero(hit & (_counts(s, m) > 0))[:, 0].split(1 << 15):  # no moments: transparent
            out[r] = _image(lam[r], lo[r], hi[r], near[r], far[r], s["table"].double(), s["rp"])
        return out.view(H, W, 4)
    if _samples(case) * m * (3 if k == "train" else 1) > (2e10 if k == "train" else 8e10):
        return None
    vox, rp, table = s["vox"], s["rp"], s["table"].double()
    o, d, near, far, hit = _rays(s["cam"], s["dmin"], s["dmax"], W, H)
    mo = torch.zeros((W * H, m), device=DEV, dtype=torch.float64)
    img = torch.zeros((W * H, 4), device=DEV, dtype=torch.float64)
    g_vox = torch.zeros(vox.numel(), device=DEV, dtype=torch.float64) if k == "train" else None
    g_table = torch.zeros_like(table)
    chunk = 1 << (12 if k == "train" else 14)
    for r in torch.nonzero(hit)[:, 0].split(chunk):
        seg = _Segments(vox, s["dmin"], s["dmax"], s["gp"], [c[r] for c in o], [c[r] for c in d], near[r], far[r],
                        keep_corners=k == "train")
        mom = seg.moments(m)
        mo[r] = mom
        if k == "generate":
            continue
        lo, hi = _quantised(seg.lo, seg.hi)
        full = torch.full((r.numel(),), m, device=DEV)
        if k == "frame":
            img[r] = _image(_multipliers(mom, rp.bias, full), lo, hi, near[r], far[r], table, rp)
            continue
        with torch.enable_grad():
            mom, tab = mom.detach().requires_grad_(), table.detach().requires_grad_()
            rgba = _image(_multipliers(mom, rp.bias, full), lo, hi, near[r], far[r], tab, rp)
            loss = ((rgba - s["target"].reshape(-1, 4)[r].double()) ** 2).sum() / (W * H * 4)
            gm, gt = torch.autograd.grad(loss, (mom, tab))
        img[r] = rgba.detach()
        g_table += gt
        gf = seg.moments_adjoint(gm)
        inside = (seg.f > 0) & (seg.f < 1)  # the clamp of the density passes no gradient outside
        gf = gf * inside
        row = 0
        for at, wt in zip(seg.at, seg.wt):
            part = gf[row:row + at.shape[1]]
            g_vox.index_add_(0, at.reshape(-1), (wt.double() * part).reshape(-1))
            row += at.shape[1]
    if k == "generate":
        return mo.view(H, W, m), None
    if k == "frame":
        return mo.view(H, W, m), None, img.view(H, W, 4)
    return img.view(H, W, 4), g_vox.view(vox.shape), g_table


def _gather64(s):
    """Kernel-weighted means of the particles closer than h to each voxel position."""
    case = s["case"]
    n, h = case["n"], _f(case["h"])
    x, y, z, v = s["parts"]
    p = [x, y, z]
    size, ext = (n, n, n // 2), (1.0, 1.0, 0.5)
    at = [0.0 + _f32div(torch.arange(k, device=DEV).float(), k) * e for k, e in zip(size, ext)]
    reach = [int(math.ceil(h / e * k)) + 1 for k, e in zip(size, ext)]
    cell = [(q.double() / e * k).floor().long() for q, e, k in zip(p, ext, size)]
    num = torch.zeros(size[0] * size[1] * size[2], device=DEV, dtype=torch.float64)
    den = torch.zeros_like(num)
    sigma, r2 = _f(0.5641895835477563), float(np.float32(h) * np.float32(h))
    for dz in range(-reach[2], reach[2] + 1):
        for dy in range(-reach[1], reach[1] + 1):
            for dx in range(-reach[0], reach[0] + 1):
                c = [a + o for a, o in zip(cell, (dx, dy, dz))]
                ok = (c[0] >= 0) & (c[0] < size[0]) & (c[1] >= 0) & (c[1] < size[1]) & (c[2] >= 0) & (c[2] < size[2])
                c = [a.clamp(0, k - 1) for a, k in zip(c, size)]
                e = [w[a] - q for w, a, q in zip(at, c, p)]
                ok &= (e[0] * e[0] + e[1] * e[1] + e[2] * e[2]) < r2  # the float test decides membership
                q = torch.nonzero(ok)[:, 0]
                if not q.numel():
                    continue
                e = [a[q].double() for a in e]
                d = (e[0] * e[0] + e[1] * e[1] + e[2] * e[2]).sqrt() / h
                w = sigma * torch.where(d < 1, 1 - 1.5 * d * d * (1 - 0.5 * d), 0.25 * (2 - d) ** 3)
                i = (c[2][q] * size[1] + c[1][q]) * size[0] + c[0][q]
                den.index_add_(0, i, w)
                num.index_add_(0, i, w * v[q].double())
    return torch.where(den != 0, num / torch.where(den != 0, den, torch.ones_like(den)), num).view(size[::-1])

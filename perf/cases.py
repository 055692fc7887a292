"""The work that users of this framework have it do, as timed cases.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare(case, seed)`` makes a case's inputs and what a program keeps
beside them, ``run(state)`` is one pass through the public entry points,
``exact(case, seed)`` is the result in 64-bit arithmetic where the outputs are
computed numbers, and ``work(case)`` the bytes and operations a pass cannot do
without.

Kinds of case:

* ``device``: one masked diffusion on device buffers (mxb_device_diffusion);
* ``host``: the Python drop-in ``maxibone_amd.diffusion.diffusion`` on numpy
  arrays, as the implant-field driver calls it;
* ``batch``: a plan over many uneven sub-volumes (capi.BatchPlan), kept and
  run again;
* ``edt`` / ``edt_field``: the distance transform and the implant EDT field;
* ``combine``: the Gaussian and EDT fields combined into one uint16 field;
* ``axis_histograms`` / ``field_histogram``: the 2D histograms of a voxel
  volume, from empty bins.
"""
import math

import numpy as np
import torch

from maxibone_amd import capi
from maxibone_amd.diffusion import diffusion

_DEV = "cuda"


def listed():
    return [
        # a try-out on a thumbnail of a scan: launches and host work only
        {"name": "diffusion_24x40x72_fp32", "kind": "device", "nz": 24, "ny": 40, "nx": 72, "sigma": 2.0,
         "reps": 3, "precision": "fp32", "out": "u16"},
        # a small region of interest
        {"name": "diffusion_128_split", "kind": "device", "nz": 128, "ny": 128, "nx": 128, "sigma": 3.0,
         "reps": 10, "precision": "fp32_split", "out": "u16"},
        # a cropped scan whose extents divide by nothing, state returned as floats
        {"name": "diffusion_ragged_fp32", "kind": "device", "nz": 257, "ny": 331, "nx": 403, "sigma": 4.0,
         "reps": 10, "precision": "fp32", "out": "f32"},
        # the implant field of a whole 1024^3 scan, at FP32 accuracy
        {"name": "diffusion_1024_split", "kind": "device", "nz": 1024, "ny": 1024, "nx": 1024, "sigma": 10.0,
         "reps": 40, "precision": "fp32_split", "out": "u16"},
        # the same in the fast 16-bit form, on rows that are not 128-byte aligned
        {"name": "diffusion_1000_bf16", "kind": "device", "nz": 1000, "ny": 1000, "nx": 1000, "sigma": 10.0,
         "reps": 20, "precision": "bf16", "out": "f32"},
        # the drop-in call of the implant-field driver on host arrays
        {"name": "drop_in_256", "kind": "host", "nz": 256, "ny": 256, "nx": 256, "sigma": 5.0, "reps": 10},
        # many uneven sub-volumes, each with its own sigma
        {"name": "batch_16_fp32", "kind": "batch", "volumes": 16, "lo": 64, "hi": 384, "reps": 20,
         "precision": "fp32"},
        # distances of a small ragged volume
        {"name": "edt_129x300x257", "kind": "edt", "nz": 129, "ny": 300, "nx": 257},
        # the EDT field of a whole scan's implant mask
        {"name": "edt_field_1024", "kind": "edt_field", "nz": 1024, "ny": 1024, "nx": 1024},
        # the two fields of a whole scan combined
        {"name": "combine_1024", "kind": "combine", "nz": 1024, "ny": 1024, "nx": 1024},
        # the histograms of a whole scan along its axes and radius
        {"name": "axis_histograms_1024", "kind": "axis_histograms", "nz": 1024, "ny": 1024, "nx": 1024,
         "voxel_bins": 4096},
        # the histogram of a whole scan against a half-resolution field
        {"name": "field_histogram_1024", "kind": "field_histogram", "nz": 1024, "ny": 1024, "nx": 1024,
         "voxel_bins": 4096, "field_bins": 2048, "field_scale": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, lo, hi, most):
    """Three extents, spread over their logarithm: a third cubes of a multiple of 8, the rest each its own."""
    while True:
        if rng.random() < 1 / 3:
            n = max(8, _log_int(rng, lo, hi) // 8 * 8)
            e = (n, n, n)
        else:
            mid = _log_int(rng, lo, hi)
            e = tuple(min(hi, max(lo, _log_int(rng, mid * 0.6, mid * 1.6))) for _ in range(3))
            if rng.random() < 0.5:
                e = (e[0], e[1], max(8, e[2] // 8 * 8))
        if e[0] * e[1] * e[2] <= most:
            return {"nz": e[0], "ny": e[1], "nx": e[2]}


def draw(rng):
    kind = rng.choice(["device"] * 6 + ["host", "batch", "edt", "edt_field", "combine", "axis_histograms",
                                        "field_histogram"])
    if kind == "device":
        e = _extents(rng, 16, 1024, 1 << 30)
        n = e["nz"] * e["ny"] * e["nx"]
        reps = min(_log_int(rng, 1, 40), max(1, int(2.4e10 / n)))
        return {"kind": kind, **e, "sigma": round(rng.uniform(1.0, 15.0), 2), "reps": reps,
                "precision": rng.choice(["fp32", "fp32_split", "fp32_split", "bf16", "bf16", "fp16"]),
                "out": rng.choice(["u16", "u16", "f32"])}
    if kind == "host":
        return {"kind": kind, **_extents(rng, 24, 512, 1 << 27), "sigma": round(rng.uniform(1.0, 10.0), 2),
                "reps": _log_int(rng, 1, 40)}
    if kind == "batch":
        lo = rng.randrange(32, 97)
        return {"kind": kind, "volumes": _log_int(rng, 2, 32), "lo": lo, "hi": rng.randrange(lo + 32, 385),
                "reps": _log_int(rng, 3, 20), "precision": rng.choice(["fp32", "bf16", "fp16"])}
    if kind == "edt":
        return {"kind": kind, **_extents(rng, 24, 640, 1 << 27)}
    case = {"kind": kind, **_extents(rng, 48, 1024, 1 << 30)}
    if kind == "axis_histograms":
        case["voxel_bins"] = rng.choice([256, 1024, 2048, 4096, 5000])
    if kind == "field_histogram":
        case.update(voxel_bins=rng.choice([256, 1024, 4096]), field_bins=rng.choice([256, 1024, 2048]),
                    field_scale=rng.choice([1, 2, 4]))
    return case


# ------------------------------------------------------------------ inputs
def _taps(sigma):
    """Gaussian taps of radius round(4 sigma), normalised in FP64, as float32."""
    r = round(4.0 * sigma)
    x = np.arange(-r, r + 1)
    phi = np.exp((-0.5 / (sigma * sigma)) * (x * x))
    return (phi / phi.sum()).astype(np.float32)


def _implant_mask(shape, seed):
    """uint8 mask on the device: a solid cylinder along z and scattered balls,
    one per ~50^3 voxels (at most 2000), of radii up to a twenty-fifth of the
    extent."""
    nz, ny, nx = shape
    rng = np.random.default_rng(seed)
    yy = (torch.arange(ny, device=_DEV) - ny // 2).view(-1, 1) ** 2
    xx = (torch.arange(nx, device=_DEV) - nx // 2).view(1, -1) ** 2
    cyl_r = int(min(ny, nx) * rng.uniform(0.15, 0.3))
    mask = (yy + xx <= cyl_r * cyl_r).to(torch.uint8).expand(nz, ny, nx).contiguous()
    size = (nz * ny * nx) ** (1 / 3)
    r_hi = max(2, int(size / 25))
    for _ in range(int(min(2000, max(4, nz * ny * nx / 5e4)))):
        c = [int(rng.integers(0, m)) for m in shape]
        r = int(rng.integers(max(1, r_hi // 6), r_hi + 1))
        lo = [max(v - r, 0) for v in c]
        hi = [min(v + r + 1, m) for v, m in zip(c, shape)]
        d = [(torch.arange(a, b, device=_DEV) - v) ** 2 for a, b, v in zip(lo, hi, c)]
        ball = d[0].view(-1, 1, 1) + d[1].view(1, -1, 1) + d[2].view(1, 1, -1) <= r * r
        mask[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] |= ball
    return mask


def _polar(ny, nx):
    y = torch.arange(ny, device=_DEV, dtype=torch.float32).view(-1, 1) - ny / 2
    x = torch.arange(nx, device=_DEV, dtype=torch.float32).view(1, -1) - nx / 2
    return torch.hypot(y, x) / (min(ny, nx) / 2), torch.atan2(y.expand(ny, nx), x.expand(ny, nx))


def _cylinder(ny, nx):
    y = torch.linspace(-1, 1, ny, device=_DEV, dtype=torch.float64).view(-1, 1)
    x = torch.linspace(-1, 1, nx, device=_DEV, dtype=torch.float64).view(1, -1)
    return (x * x + y * y < 1).to(torch.uint8).contiguous()


def _rod_mask(shape, seed):
    """uint8 implant mask on the device: a threaded rod along z from a quarter
    of the depth on, and scattered bright specks."""
    nz, ny, nx = shape
    g = torch.Generator(device=_DEV).manual_seed(seed)
    turn, start = torch.rand(2, generator=g, device=_DEV).tolist()
    r, phi = _polar(ny, nx)
    m = torch.zeros(shape, dtype=torch.uint8, device=_DEV)
    for z in range(int(nz * (0.2 + 0.1 * start)), nz):
        m[z] = r < 0.12 + 0.015 * torch.sin(phi + 2 * math.pi * (z / 48.0 + turn))
    at = torch.randint(0, m.numel(), (max(1, m.numel() // 200000),), generator=g, device=_DEV)
    m.view(-1)[at] = 1
    return m


def _u16(t):
    """uint16 bits of a float tensor's values, clipped, in an int16 tensor."""
    return t.clamp_(0, 65535).to(torch.int32).to(torch.int16)


def _ct_voxels(shape, seed):
    """CT-like uint16 voxels: material classes by radius (implant, bone, soft
    tissue, air) with noise."""
    nz, ny, nx = shape
    g = torch.Generator(device=_DEV).manual_seed(seed)
    r, _ = _polar(ny, nx)
    base = torch.where(r < 0.15, 52000.0, torch.where(r < 0.45, 24000.0, torch.where(r < 0.9, 9000.0, 1500.0)))
    v = torch.empty(shape, dtype=torch.int16, device=_DEV)
    for z in range(0, nz, 32):
        m = min(32, nz - z)
        v[z:z + m] = _u16(torch.randn((m, ny, nx), generator=g, device=_DEV) * 700.0 + base)
    return v


def _smooth_fields(shape, seed):
    """The Gaussian and the EDT field of a rod: smooth, decaying from the
    axis, slowly varying along it."""
    nz, ny, nx = shape
    rng = np.random.default_rng(seed)
    rad, phase = 0.1 + 0.1 * rng.random(), 6.28 * rng.random()
    r, _ = _polar(ny, nx)
    gauss2 = 65535.0 * torch.exp(-(r - rad).clamp(min=0) * 6)
    edt2 = (r - rad).abs() * 40000.0
    gauss = torch.empty(shape, dtype=torch.int16, device=_DEV)
    edt = torch.empty(shape, dtype=torch.int16, device=_DEV)
    for z in range(nz):
        gauss[z] = _u16(gauss2 * (1.0 + 0.1 * math.sin(z / 37.0 + phase)))
        edt[z] = _u16(edt2 * (1.0 + 0.05 * math.sin(z / 23.0 + phase)))
    return gauss, edt


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device=_DEV)


def _output(shape, kind):
    """An output volume; uint16 values as the bits of int16, which torch can index."""
    return torch.empty(shape, dtype=torch.int16 if kind == "u16" else torch.float32, device=_DEV)


def _batch_shapes(case, seed):
    """Shapes and sigmas of a batch: the same for every seed, so that a pass is the same work."""
    rng = np.random.default_rng([case["volumes"], case["lo"], case["hi"], 5])
    return [(tuple(int(v) for v in rng.integers(case["lo"], case["hi"] + 1, 3)), float(rng.uniform(2.0, 10.0)))
            for _ in range(case["volumes"])]


def prepare(case, seed):
    kind, L = case["kind"], capi.lib()
    s = {"case": case}
    if kind == "batch":
        vols = _batch_shapes(case, seed)
        s["masks"] = [_implant_mask(shape, seed * 1000 + i) for i, (shape, _) in enumerate(vols)]
        s["outs"] = [_output(shape, "u16") for shape, _ in vols]
        torch.cuda.synchronize()  # the plan runs on a stream of its own
        s["plan"] = capi.BatchPlan([m.data_ptr() for m in s["masks"]], [shape for shape, _ in vols],
                                   [_taps(sigma) for _, sigma in vols], case["reps"],
                                   outs_u16=[o.data_ptr() for o in s["outs"]], precision=case["precision"],
                                   stream=_stream() or None)
        return s
    shape = (case["nz"], case["ny"], case["nx"])
    if kind in ("device", "host"):
        s["taps"] = _taps(case["sigma"])
        s["mask"] = _implant_mask(shape, seed)
        if kind == "host":
            s["mask"] = s["mask"].cpu().numpy()
            s["out"] = np.zeros(shape, np.uint16)
            return s
        size = L.mxb_state_bytes(capi.PRECISION[case["precision"]], *shape)
        s["state"] = [_bytes(size), _bytes(size)]
        s["out"] = _output(shape, case["out"])
    elif kind in ("edt", "edt_field"):
        m = _rod_mask(shape, seed)
        s["mask"] = m if kind == "edt_field" else (m == 0).to(torch.uint8)  # edt: distance to the nearest zero
        s["ws"] = _bytes(L.mxb_edt_workspace_bytes(*shape))
        s["cyl"] = _cylinder(*shape[1:])
        s["out"] = _output(shape, "u16" if kind == "edt_field" else "f32")
    elif kind == "combine":
        s["gauss"], s["edt"] = _smooth_fields(shape, seed)
        s["cyl"] = _cylinder(*shape[1:])
        s["ws"] = _bytes(L.mxb_combine_workspace_bytes())
        s["out"] = _output(shape, "u16")
    else:
        s["voxels"] = _ct_voxels(shape, seed)
        s["ws"] = _bytes(L.mxb_histogram_workspace_bytes(*shape))
        vb = case["voxel_bins"]
        if kind == "field_histogram":
            k = case["field_scale"]
            s["field"] = _smooth_fields(shape, seed)[0][::k, ::k, ::k].contiguous()
            s["bins"] = [torch.zeros((case["field_bins"], vb), dtype=torch.int64, device=_DEV)]
        else:
            s["radii"] = int(math.hypot(shape[1] - shape[1] // 2, shape[2] - shape[2] // 2)) + 1
            s["bins"] = [torch.zeros((m, vb), dtype=torch.int64, device=_DEV)
                         for m in (shape[2], shape[1], shape[0], s["radii"])]
    return s


# ------------------------------------------------------------------ a pass
_VRANGE, _FRANGE = (1.0, 40000.0), (1.0, 65535.0)


def run(s):
    case = s["case"]
    kind, L = case["kind"], capi.lib()
    if kind == "batch":
        s["plan"].run()
        return s["outs"]
    shape = (case["nz"], case["ny"], case["nx"])
    if kind == "host":
        diffusion(s["mask"], s["taps"], s["out"], case["reps"])
        return s["out"]
    if kind == "device":
        u16 = s["out"].data_ptr() if case["out"] == "u16" else None
        f32 = s["out"].data_ptr() if case["out"] == "f32" else None
        capi.check(L.mxb_device_diffusion(s["mask"].data_ptr(), *shape, s["taps"].ctypes.data, s["taps"].size,
                                          case["reps"], capi.PRECISION[case["precision"]],
                                          s["state"][0].data_ptr(), s["state"][1].data_ptr(), u16, f32, _stream()))
        return s["out"]
    if kind == "edt":
        capi.check(L.mxb_device_edt(s["mask"].data_ptr(), *shape, None, s["out"].data_ptr(), s["ws"].data_ptr(),
                                    _stream()))
        return s["out"]
    if kind == "edt_field":
        capi.check(L.mxb_device_edt_field(s["mask"].data_ptr(), *shape, s["cyl"].data_ptr(), s["out"].data_ptr(),
                                          s["ws"].data_ptr(), _stream()))
        return s["out"]
    if kind == "combine":
        capi.check(L.mxb_device_combine_fields(s["gauss"].data_ptr(), s["edt"].data_ptr(), *shape,
                                               s["cyl"].data_ptr(), s["out"].data_ptr(), s["ws"].data_ptr(),
                                               _stream()))
        return s["out"]
    for b in s["bins"]:
        b.zero_()
    if kind == "field_histogram":
        capi.check(L.mxb_device_field_histogram(s["voxels"].data_ptr(), *shape, s["field"].data_ptr(),
                                                *s["field"].shape, s["bins"][0].data_ptr(), case["field_bins"],
                                                case["voxel_bins"], *_VRANGE, *_FRANGE, s["ws"].data_ptr(),
                                                _stream()))
    else:
        capi.check(L.mxb_device_axis_histograms(s["voxels"].data_ptr(), *shape, 0, *(b.data_ptr() for b in s["bins"]),
                                                shape[0], s["radii"], case["voxel_bins"], shape[1] // 2,
                                                shape[2] // 2, *_VRANGE, s["ws"].data_ptr(), _stream()))
    return s["bins"]


# ------------------------------------------------------------------ results in 64 bits
def _toeplitz(n, taps):
    """T with (T u)[i] = sum_r taps[R + r] u[i + r], zero outside [0, n)."""
    R = taps.shape[0] // 2
    i = torch.arange(n, device=_DEV)
    d = i.view(1, -1) - i.view(-1, 1) + R
    inside = (d >= 0) & (d <= 2 * R)
    return torch.where(inside, taps[d.clamp(0, 2 * R)], torch.zeros((), dtype=taps.dtype, device=_DEV)).contiguous()


def exact(case, seed):
    if case["kind"] == "device" and case["out"] == "f32":
        nz, ny, nx = shape = (case["nz"], case["ny"], case["nx"])
        mask = _implant_mask(shape, seed) > 0
        taps = torch.from_numpy(_taps(case["sigma"])).to(_DEV, torch.float64)
        tz, ty, tx = (_toeplitz(m, taps) for m in shape)
        tx = tx.t().contiguous()
        u = mask.to(torch.float64)
        for _ in range(case["reps"]):
            u = torch.mm(tz, u.view(nz, ny * nx)).view(shape)
            for z in range(nz):
                u[z] = torch.mm(torch.mm(ty, u[z]), tx)
            u[mask] = 1.0
        return u
    if case["kind"] == "edt":
        shape = (case["nz"], case["ny"], case["nx"])
        m = _rod_mask(shape, seed) == 0
        d = torch.where(m, torch.full((), 1e12, dtype=torch.float64, device=_DEV),
                        torch.zeros((), dtype=torch.float64, device=_DEV))
        for axis in (2, 1, 0):
            g = d.movedim(axis, 0)
            best = g.clone()
            for k in range(1, shape[axis]):
                torch.minimum(best[k:], g[:-k] + float(k * k), out=best[k:])
                torch.minimum(best[:-k], g[k:] + float(k * k), out=best[:-k])
            d = best.movedim(0, axis).contiguous()
        return d.sqrt()
    return None  # whole numbers


def work(case):
    """Each input read once and each output written once; two operations per
    tap, axis and repetition of a diffusion."""
    kind = case["kind"]
    if kind == "batch":
        flops = data = 0.0
        for shape, sigma in _batch_shapes(case, 0):
            n = float(np.prod(shape))
            flops += 6.0 * _taps(sigma).size * case["reps"] * n
            data += 3.0 * n
        return {"bytes": data, "flops": flops}
    n = float(case["nz"]) * case["ny"] * case["nx"]
    if kind in ("device", "host"):
        out = 4 if case.get("out") == "f32" else 2
        return {"bytes": (1.0 + out) * n, "flops": 6.0 * _taps(case["sigma"]).size * case["reps"] * n}
    if kind == "field_histogram":
        return {"bytes": (2.0 + 2.0 / case["field_scale"] ** 3) * n + 8.0 * case["field_bins"] * case["voxel_bins"],
                "flops": 0.0}
    if kind == "axis_histograms":
        lines = case["nx"] + case["ny"] + case["nz"] + math.hypot(case["ny"], case["nx"]) / 2
        return {"bytes": 2.0 * n + 8.0 * lines * case["voxel_bins"], "flops": 0.0}
    return {"bytes": {"edt": 5.0, "edt_field": 3.0, "combine": 6.0}[kind] * n, "flops": 0.0}

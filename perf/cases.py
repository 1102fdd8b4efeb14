"""Cases that stand for what a program has this framework do, and how to run each.

Every case is one pass through public entry points of ``fdk_amd``: whole small
reconstructions, backprojection passes over mirror slab pairs, boxes and full
volumes, the row filter, the ray-marching projector, one multiplicative update of
the iterative loop, the RTK-form backprojector, and the U-Net's layers (forward,
decoder form, backward).  ``listed()`` names representative sizes, ``draw()``
samples the same ranges, ``exact()`` restates each case in 64 bits with plain
torch and numpy.
"""
import math

import numpy as np
import torch

import fdk_amd as F
from fdk_amd import iterative, learned
from fdk_amd import unet as U

SOD, SID = 1000.0, 1500.0
DEV = "cuda"
NPDT = {"f32": F.FDK_F32, "f16": F.FDK_F16, "bf16": F.FDK_BF16}
TDT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # The smallest whole reconstruction (the package's smoke size): filter, two
        # 32-view passes, handle and all.  Launches and host work count here.
        {"name": "fdk_64", "kind": "fdk", "n": 64, "views": 64},
        # The 256^3 scan of the reference's own tests, a mirror slab pair, FP32 views.
        {"name": "bp_pair_256", "kind": "bp", "nx": 256, "ny": 256, "nz": 256, "nu": 256, "nv": 256,
         "views": 96, "dtype": "f32", "box": "pair", "transpose": 1},
        # A whole 1024^3 volume from FP16 views of 1024^2: the large end.
        {"name": "bp_pair_1024_f16", "kind": "bp", "nx": 1024, "ny": 1024, "nz": 1024, "nu": 1024,
         "nv": 1024, "views": 64, "dtype": "f16", "box": "pair", "transpose": 1},
        # A 256^3 region off the centre of a 1024^3 scan, as training pairs are cut.
        {"name": "bp_box_256", "kind": "bp", "nx": 1024, "ny": 1024, "nz": 1024, "nu": 1024,
         "nv": 1024, "views": 128, "dtype": "f32", "box": "box", "ox": 200, "oy": 310, "oz": 270,
         "w": 256, "h": 256, "d": 256, "transpose": 1},
        # One multiplicative update at odd sizes: projector, u-fastest views into a
        # full volume without a mirror slab, and the loop's own arithmetic.
        {"name": "ratio_odd", "kind": "ratio", "nx": 101, "ny": 92, "nz": 83, "nu": 121, "nv": 98,
         "views": 40},
        # One 32-view batch of 2048^2 raw views, filtered and transposed, FP32.
        {"name": "filter_2048", "kind": "filter", "nu": 2048, "nv": 2048, "views": 32,
         "dtype": "f32", "pad": 4, "transpose": 1},
        # Views of 4096^2 filtered (N = 8192) into FP16 storage with per-view scales.
        {"name": "filter_4096_f16", "kind": "filter", "nu": 4096, "nv": 4096, "views": 8,
         "dtype": "f16", "pad": 4, "transpose": 1},
        # Ray marching through 256^3 with half-voxel steps, views all round the scan.
        {"name": "fp_256", "kind": "fp", "nx": 256, "ny": 256, "nz": 256, "nu": 256, "nv": 256,
         "views": 24, "step": 0.5, "mode": 0},
        # The RTK call of the reference: one 32-view pass, u-fastest views.
        {"name": "rtk_384", "kind": "rtk", "nx": 384, "ny": 384, "nz": 320, "nu": 512, "nv": 480,
         "views": 32},
        # The middle level of the edge-4 network on a 1024^3 volume.
        {"name": "conv_64", "kind": "conv", "cin": 64, "cout": 64, "cup": 0, "n": 1, "d": 128,
         "h": 128, "w": 128},
        # The last decoder's first layer, [upsampled 64, skip 32] -> 32, on half its grid.
        {"name": "conv_cat", "kind": "conv", "cin": 96, "cout": 32, "cup": 64, "n": 1, "d": 128,
         "h": 256, "w": 256},
        # A full-width layer's backward at the edge-4 network's training shape.
        {"name": "conv_bwd", "kind": "conv_bwd", "cin": 32, "cout": 32, "n": 4, "d": 64, "h": 64,
         "w": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fdk", "bp", "bp", "bp", "ratio", "filter", "filter", "fp", "rtk", "conv",
                       "conv_bwd"])
    if kind == "fdk":
        return {"kind": kind, "n": 2 * _log(rng, 24, 96), "views": _log(rng, 20, 200)}
    if kind == "bp":
        n = _log(rng, 64, 512)
        c = {"kind": kind, "nx": n + rng.randrange(-8, 9), "ny": n + rng.randrange(-8, 9),
             "nz": n + rng.randrange(-8, 9), "nu": n + rng.randrange(-4, 60),
             "nv": n + rng.randrange(-4, 60), "views": _log(rng, 8, 128),
             "dtype": rng.choice(["f32", "f32", "f16", "bf16"]),
             "box": rng.choice(["pair", "pair", "box", "full"]), "transpose": 1}
        if rng.random() < 0.6:  # detectors usually come in multiples of 4
            c["nu"], c["nv"] = c["nu"] // 4 * 4, c["nv"] // 4 * 4
        if c["box"] == "full" and c["dtype"] == "f32":
            c["transpose"] = rng.choice([0, 1])
        if c["box"] == "pair":
            c["nz"] -= c["nz"] % 2
        if c["box"] == "box":
            for o, s, m in (("ox", "w", "nx"), ("oy", "h", "ny"), ("oz", "d", "nz")):
                c[s] = rng.randrange(c[m] // 4, c[m] // 2 + 1)
                c[o] = rng.randrange(0, c[m] - c[s] + 1)
        return c
    if kind == "ratio":
        n = _log(rng, 48, 128)
        return {"kind": kind, "nx": n + rng.randrange(9), "ny": n + rng.randrange(9),
                "nz": n + rng.randrange(9), "nu": n + rng.randrange(8, 40),
                "nv": n + rng.randrange(8, 40), "views": _log(rng, 12, 64)}
    if kind == "filter":
        nu = _log(rng, 128, 2900)
        nv = max(64, min(3000, int(nu * rng.uniform(0.6, 1.2))))
        if rng.random() < 0.6:
            nu, nv = nu // 4 * 4, nv // 4 * 4
        return {"kind": kind, "nu": nu, "nv": nv,
                "views": max(1, min(_log(rng, 4, 64), int(1.3e8 / (nu * nv)))),
                "dtype": rng.choice(["f32", "f32", "f16", "bf16"]), "pad": rng.choice([4, 4, 3, 0]),
                "transpose": rng.choice([1, 1, 1, 0])}
    if kind == "fp":
        n = _log(rng, 64, 320)
        return {"kind": kind, "nx": n + rng.randrange(9), "ny": n + rng.randrange(9),
                "nz": n + rng.randrange(9), "nu": n + rng.randrange(60), "nv": n + rng.randrange(60),
                "views": _log(rng, 1, 24), "step": rng.choice([0.0, 0.5]),
                "mode": rng.choice([0, 1])}
    if kind == "rtk":
        n = _log(rng, 64, 400)
        return {"kind": kind, "nx": n + rng.randrange(9), "ny": n + rng.randrange(9),
                "nz": n + rng.randrange(9), "nu": n + rng.randrange(100),
                "nv": n + rng.randrange(100), "views": _log(rng, 4, 32)}
    if kind == "conv":
        cin, cout, cup = rng.choice([(32, 32, 0), (32, 64, 0), (64, 64, 0), (64, 128, 0),
                                     (128, 128, 0), (192, 64, 128), (96, 32, 64)])
        return {"kind": kind, "cin": cin, "cout": cout, "cup": cup, "n": rng.choice([1, 2, 4]),
                "d": 4 * rng.randrange(2, 9), "h": 16 * rng.randrange(1, 9),
                "w": 32 * rng.randrange(1, 7)}
    cin, cout = rng.choice([(32, 32), (32, 64), (64, 64), (64, 128), (128, 128)])
    return {"kind": kind, "cin": cin, "cout": cout, "n": rng.choice([1, 2, 4]),
            "d": 4 * rng.randrange(2, 9), "h": 16 * rng.randrange(1, 5),
            "w": 32 * rng.randrange(1, 5)}


# ------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) + 1)
    return g


def _para(c):
    """A scan whose detector just covers the volume (1.5x magnification)."""
    if c["kind"] == "fdk":
        return learned.geometry(c["n"], c["views"])
    n = max(c["nx"], c["ny"], c["nz"])
    vox = 256.0 / n
    return F.Parameter(nx=c["nx"], ny=c["ny"], nz=c["nz"], dx=vox, dy=vox, dz=vox, nu=c["nu"],
                       nv=c["nv"], du=1.62 * vox * n / c["nu"], dv=1.62 * vox * n / c["nv"],
                       sod=SOD, sid=SID, nproj=c["views"], direction=-1, scan_angle_deg=360.0,
                       volume_position_angle_rad=0.0, filter_type=5)


def _spheres(p, g, count=10):
    """Random spheres inside the volume: (count, 5) of centre, radius, density."""
    fov = min(p.nx * p.dx, p.ny * p.dy)
    r = torch.rand((count, 5), generator=g, device=DEV, dtype=torch.float64)
    s = torch.empty_like(r)
    s[:, 3] = fov * (0.04 + 0.16 * r[:, 3])
    ang, rad = 2 * math.pi * r[:, 0], (0.45 * fov - s[:, 3]) * r[:, 1].sqrt()
    s[:, 0], s[:, 1] = rad * ang.cos(), rad * ang.sin()
    s[:, 2] = (r[:, 2] - 0.5) * 0.7 * p.nz * p.dz
    s[:, 4] = 0.2 + 0.8 * r[:, 4]
    return s


def _theta(p):
    deg = np.arange(p.nproj) * p.scan_angle_deg / p.nproj
    return p.direction * deg / 180.0 * math.pi + p.volume_position_angle_rad


def _line_integrals(p, s, noise, g):
    """Views (nproj, nv, nu) of the spheres' chord lengths, with a little noise."""
    out = torch.empty((p.nproj, p.nv, p.nu), device=DEV)
    um = (torch.arange(p.nu, device=DEV, dtype=torch.float64) - (p.nu - 1) / 2) * p.du
    vm = (torch.arange(p.nv, device=DEV, dtype=torch.float64) - (p.nv - 1) / 2) * -p.dv
    nrm = torch.rsqrt(um[None, :] ** 2 + vm[:, None] ** 2 + p.sid ** 2)
    cen = s.cpu().numpy()
    for q, th in enumerate(_theta(p)):
        acc = torch.zeros((p.nv, p.nu), device=DEV)
        for x, y, z, r, rho in cen:
            a, b = x * math.cos(th) - y * math.sin(th), x * math.sin(th) + y * math.cos(th) + p.sod
            t = (a * um[None, :] + b * p.sid + z * vm[:, None]) * nrm
            d2 = a * a + b * b + z * z - t * t
            acc += (2 * rho * torch.sqrt(torch.clamp(r * r - d2, min=0.0))).float()
        out[q] = acc
    if noise:
        out += noise * torch.randn(out.shape, generator=g, device=DEV)
    return out


def _filtered(p, g):
    """Ramp-filtered noisy views, transposed (nproj, nu, nv): what a backprojector meets."""
    raw = _line_integrals(p, _spheres(p, g, 4), 0.5, g)
    n = 2 * p.nu
    ramp = torch.linspace(0, 1, n // 2 + 1, device=DEV) * 0.05
    out = torch.empty((p.nproj, p.nu, p.nv), device=DEV)
    for q in range(p.nproj):
        f = torch.fft.irfft(torch.fft.rfft(raw[q], n=n) * ramp, n=n)[:, :p.nu]
        out[q] = f.t()
    return out


def _boxes(c):
    if c["box"] == "pair":
        h = c["nz"] // 2
        return (0, 0, 0, c["nx"], c["ny"], h), (0, 0, h, c["nx"], c["ny"], h)
    if c["box"] == "box":
        return (c["ox"], c["oy"], c["oz"], c["w"], c["h"], c["d"]), (0, 0, 0, 0, 0, 0)
    return (0, 0, 0, c["nx"], c["ny"], c["nz"]), (0, 0, 0, 0, 0, 0)


def _bp_inputs(c, seed):
    """Stored views, their scale/offset (16-bit) and the scan."""
    p = _para(c)
    v = _filtered(p, _gen(seed))
    if c["dtype"] == "f32":
        return p, (v.transpose(1, 2).contiguous() if not c["transpose"] else v), None
    lo = v.amin(dim=(1, 2))
    sc = v.amax(dim=(1, 2)) - lo
    q = ((v - lo[:, None, None]) / sc[:, None, None]).to(TDT[c["dtype"]])
    return p, q, torch.stack([sc, lo], 1).cpu().numpy()


def _filter_inputs(c, seed):
    g = _gen(seed)
    p = F.Parameter(nx=64, ny=64, nz=64, dx=400.0 / 96, dy=400.0 / 96, dz=400.0 / 96, nu=c["nu"],
                    nv=c["nv"], du=400.0 / c["nu"], dv=400.0 / c["nv"], sod=SOD, sid=SID,
                    nproj=c["views"], filter_type=5)
    raw = _line_integrals(p, _spheres(p, g, 3), 0.5, g)
    um = (torch.arange(p.nu, device=DEV, dtype=torch.float64) - (p.nu - 1) / 2) * p.du
    vm = (torch.arange(p.nv, device=DEV, dtype=torch.float64) - (p.nv - 1) / 2) * p.dv
    cos = (SID * torch.rsqrt(um[None, :] ** 2 + vm[:, None] ** 2 + SID ** 2)).float()
    n = 1 << int(c["nu"]).bit_length()
    k = torch.arange(n, device=DEV, dtype=torch.float64)
    k = torch.minimum(k, n - k)
    H = (2 * k / n * 0.5 * (1 + torch.cos(2 * math.pi * k / n))).float()
    return raw, cos, H


def _volume(p, g):
    """A volume of soft-edged spheres with a little noise, (nz, ny, nx)."""
    s = _spheres(p, g).cpu().numpy()
    x = (torch.arange(p.nx, device=DEV) - (p.nx - 1) / 2) * p.dx
    y = -(torch.arange(p.ny, device=DEV) - (p.ny - 1) / 2) * p.dy
    z = -(torch.arange(p.nz, device=DEV) - (p.nz - 1) / 2) * p.dz
    v = 0.02 * torch.rand((p.nz, p.ny, p.nx), generator=g, device=DEV)
    for a, b, d, r, rho in s:
        q = torch.sqrt((x - a)[None, None, :] ** 2 + (y - b)[None, :, None] ** 2
                       + (z - d)[:, None, None] ** 2)
        v += rho * torch.clamp((r - q) / p.dx + 0.5, 0.0, 1.0)
    return v


def _bf16(shape, g, scale=0.5):
    return (torch.randn(shape, device=DEV, generator=g) * scale).bfloat16()


def _conv_inputs(c, seed):
    """Layer inputs, weights (27, cout, cin) and bias; activations are post-ReLU."""
    g = _gen(seed)
    s, k = (c["n"], c["d"], c["h"], c["w"]), c["cin"] - c["cup"]
    x = _bf16(s + (k,), g).relu_()
    up = _bf16((s[0], s[1] // 2, s[2] // 2, s[3] // 2, c["cup"]), g).relu_() if c["cup"] else None
    w = _bf16((27, c["cout"], c["cin"]), g, math.sqrt(2.0 / (27 * c["cin"])))
    b = 0.1 * torch.randn(c["cout"], device=DEV, generator=g)
    return x, up, w, b


def _bwd_inputs(c, seed):
    """A layer's input, output (both post-ReLU), output gradient and weights."""
    g = _gen(seed)
    s = (c["n"], c["d"], c["h"], c["w"])
    x, y = _bf16(s + (c["cin"],), g).relu_(), _bf16(s + (c["cout"],), g).relu_()
    dy = _bf16(s + (c["cout"],), g, 1e-3)
    w = _bf16((27, c["cout"], c["cin"]), g, math.sqrt(2.0 / (27 * c["cin"])))
    return x, y, dy, w


def _layer(c, w, b):
    cv = U.Conv3(c["cin"], c["cout"], 1, np.random.default_rng(0), DEV)
    cv.w.copy_(w.float())
    if b is not None:
        cv.b.copy_(b)
    cv.refresh()
    return cv


def prepare(case, seed):
    c, k = case, case["kind"]
    if k == "fdk":
        sc = learned.Scanner(_para(c))
        g = _gen(seed)
        raw = _line_integrals(sc.p, _spheres(sc.p, g), 0.5, g)
        sc.tables(c["views"])
        return {"case": c, "scanner": sc, "raw": raw,
                "store": torch.empty((c["views"], sc.p.nu, sc.p.nv), device=DEV)}
    if k == "bp":
        p, views, so = _bp_inputs(c, seed)
        top, bot = _boxes(c)
        h = F.BackProjectionFDK(p.nv, p.nu, 32, p.nx, p.ny, p.nz, top, bot)
        h.set_stream(torch.cuda.current_stream().cuda_stream)
        out = torch.empty((h.depth, top[4], top[3]), device=DEV)
        return {"case": c, "bp": h, "views": views, "so": so, "out": out, "p": p,
                "mats": p.proj_matrices().astype(np.float32)}
    if k == "ratio":
        p = _para(c)
        g = _gen(seed)
        return {"case": c, "p": p, "proj": _line_integrals(p, _spheres(p, g), 0.0, g),
                "projector": iterative.Projector(p)}
    if k == "filter":
        raw, cos, H = _filter_inputs(c, seed)
        shape = (c["views"], c["nu"], c["nv"]) if c["transpose"] else tuple(raw.shape)
        return {"case": c, "raw": raw, "cos": cos, "H": H,
                "out": torch.empty(shape, dtype=TDT[c["dtype"]], device=DEV)}
    if k == "fp":
        p = _para(c)
        return {"case": c, "p": p, "vol": _volume(p, _gen(seed)),
                "out": torch.empty((c["views"], p.nv, p.nu), device=DEV)}
    if k == "rtk":
        p = _para(c)
        g = _gen(seed)
        views = _filtered(p, g).transpose(1, 2).contiguous()
        vin = 1e-5 * torch.randn((p.nz, p.ny, p.nx), generator=g, device=DEV)
        return {"case": c, "p": p, "views": views, "vin": vin, "out": torch.empty_like(vin),
                "mats": p.proj_matrices().astype(np.float32)}
    if k == "conv":
        x, up, w, b = _conv_inputs(c, seed)
        return {"case": c, "x": x.view(torch.int16),
                "up": up.view(torch.int16) if up is not None else None, "layer": _layer(c, w, b)}
    x, y, dy, w = _bwd_inputs(c, seed)
    return {"case": c, "x": x.view(torch.int16), "y": y.view(torch.int16),
            "dy": dy.view(torch.int16), "layer": _layer(c, w, None)}


def run(state):
    c = state["case"]
    k = c["kind"]
    if k == "fdk":
        return state["scanner"].fdk(state["raw"], store=state["store"])
    if k == "bp":
        h, p, so = state["bp"], state["p"], state["so"]
        w, hh = (p.nv, p.nu) if c["transpose"] else (p.nu, p.nv)
        h.zero()
        for b in range(0, c["views"], 32):
            n = min(32, c["views"] - b)
            h.bp_device(state["views"], w, hh, state["mats"][b:b + n], n, transpose=c["transpose"],
                        dtype=NPDT[c["dtype"]], offset_views=b,
                        scale_offset=so[b:b + n] if so is not None else None)
        return h.get_volume_device(state["out"])
    if k == "ratio":
        return iterative.ratio_reconstruct(state["p"], state["proj"], 1,
                                           projector=state["projector"])
    if k == "filter":
        so = F.filter_views(state["raw"], state["out"], state["cos"], state["H"], c["pad"],
                            bool(c["transpose"]), NPDT[c["dtype"]])
        return {"views": state["out"]} if so is None else {"views": state["out"], "so": so}
    if k == "fp":
        F.forward_project(state["p"], state["vol"], 0, c["views"], state["out"], c["step"],
                          c["mode"])
        return state["out"]
    if k == "rtk":
        p = state["p"]
        F.reconstruct_conebeam((p.nu, p.nv, c["views"]), (p.nx, p.ny, p.nz), state["mats"],
                               state["vin"], state["out"], state["views"])
        return state["out"]
    cv, s = state["layer"], (c["n"], c["d"], c["h"], c["w"])
    if k == "conv":
        y = (cv.forward_cat(state["up"], c["cup"], state["x"], s) if c["cup"]
             else cv.forward(state["x"], s))
        return y.view(torch.bfloat16)
    cv.gw.zero_()
    cv.gb.zero_()
    dx = cv.backward(state["dy"], state["x"], state["y"], s)
    return {"dx": dx.view(torch.bfloat16), "gw": cv.gw, "gb": cv.gb}


def work(case):
    c, k = case, case["kind"]
    if k == "fdk":
        n, v = c["n"], c["views"]
        return {"bytes": 4.0 * (v * n * n + n ** 3),
                "flops": 8.0 * v * n ** 3 + 20.0 * v * n * n * math.log2(2 * n)}
    if k == "bp":
        t, b = _boxes(c)
        nvox = t[3] * t[4] * (t[5] + b[5])
        s = 4 if c["dtype"] == "f32" else 2
        return {"bytes": 4.0 * nvox + s * c["views"] * c["nu"] * c["nv"],
                "flops": 8.0 * c["views"] * nvox}
    if k == "ratio":
        nvox, px = c["nx"] * c["ny"] * c["nz"], c["views"] * c["nu"] * c["nv"]
        # the update's and the norm's backprojection, and one forward projection
        return {"bytes": 4.0 * (px + nvox),
                "flops": 16.0 * c["views"] * nvox + 20.0 * px * max(c["nx"], c["ny"]) * 0.6}
    if k == "filter":
        px = c["views"] * c["nu"] * c["nv"]
        n = 1 << int(c["nu"]).bit_length()
        return {"bytes": px * (4.0 + (4 if c["dtype"] == "f32" else 2)) + 4.0 * c["nu"] * c["nv"],
                "flops": 5.0 * c["views"] * c["nv"] * n * math.log2(n)}
    if k == "fp":
        px = c["views"] * c["nu"] * c["nv"]
        vox = 256.0 / max(c["nx"], c["ny"], c["nz"])
        return {"bytes": 4.0 * (c["nx"] * c["ny"] * c["nz"] + px),
                "flops": 20.0 * px * 160.0 / (c["step"] or vox)}
    if k == "rtk":
        nvox = c["nx"] * c["ny"] * c["nz"]
        return {"bytes": 8.0 * nvox + 4.0 * c["views"] * c["nu"] * c["nv"],
                "flops": 12.0 * c["views"] * nvox}
    vox = c["n"] * c["d"] * c["h"] * c["w"]
    mac = 54.0 * c["cin"] * c["cout"]
    if k == "conv":
        return {"bytes": 2.0 * vox * (c["cin"] - c["cup"] + c["cup"] / 8 + c["cout"])
                + 2.0 * 27 * c["cin"] * c["cout"], "flops": mac * vox}
    return {"bytes": 2.0 * vox * (2 * c["cin"] + 2 * c["cout"]) + 6.0 * 27 * c["cin"] * c["cout"],
            "flops": 2 * mac * vox}


# ------------------------------------------------------------------- 64-bit answers
def _mats64(p):
    """(nproj, 12) matrices (x, y, z, 1) -> (u w, v w, w) of the circular scan."""
    out = np.empty((p.nproj, 3, 4))
    cx, cy, cz = (p.nx - 1) / 2, (p.ny - 1) / 2, (p.nz - 1) / 2
    for q, th in enumerate(_theta(p)):
        c, s = math.cos(th), math.sin(th)
        w = np.array([s * p.dx, -c * p.dy, 0, p.sod - s * p.dx * cx + c * p.dy * cy])
        x = np.array([c * p.dx, s * p.dy, 0, -c * p.dx * cx - s * p.dy * cy])
        z = np.array([0, 0, p.dz, -p.dz * cz])
        out[q] = (p.sid / p.du * x + (p.nu - 1) / 2 * w, p.sid / p.dv * z + (p.nv - 1) / 2 * w, w)
    return out.reshape(-1, 12)


def _back64(view, mats, xs, ys, zs):
    """Sum over views of bilinear(view(q))[u, v] / w^2 on the grid, (len(zs), len(ys), len(xs));
    view(q): (nu, nv) FP64."""
    f64 = dict(device=DEV, dtype=torch.float64)
    x, y, z = (torch.as_tensor(np.asarray(a, np.float64), device=DEV) for a in (xs, ys, zs))
    out = torch.zeros((len(zs), len(ys), len(xs)), **f64)
    step = max(1, int(1.3e8 // (len(ys) * len(xs))))
    for q in range(mats.shape[0]):
        m, P = mats[q], view(q)
        H, W = P.shape
        flat = P.reshape(-1)
        w = m[8] * x[None, :] + m[9] * y[:, None] + m[11]
        u = (m[0] * x[None, :] + m[1] * y[:, None] + m[3]) / w
        vb = (m[4] * x[None, :] + m[5] * y[:, None] + m[7]) / w
        dv = m[6] / w
        iu = torch.floor(u)
        uok = (iu >= 0) & (iu <= H - 2)
        fu = u - iu
        row = torch.where(uok, iu, torch.zeros_like(iu)).long() * W
        zero = torch.zeros((), **f64)
        w0, w1 = torch.where(uok, (1 - fu) / w ** 2, zero), torch.where(uok, fu / w ** 2, zero)
        for a in range(0, len(zs), step):
            v = vb[None] + z[a:a + step, None, None] * dv[None]
            iv = torch.floor(v)
            v -= iv
            ok = (iv >= 0) & (iv <= W - 2)
            i = torch.where(ok, iv, zero).long()
            del iv
            i += row[None]
            lo = w0[None] * flat[i] + w1[None] * flat[i + W]
            i += 1
            hi = w0[None] * flat[i] + w1[None] * flat[i + W]
            del i
            hi -= lo
            out[a:a + step] += torch.where(ok, lo.addcmul_(v, hi), zero)
    return out


def _filter64(raw, cos, H, pad):
    """Cos weight, edge padding to len(H), multiply, crop; one (nv, nu) view."""
    x = raw.double() * cos.double()
    nu, n = x.shape[-1], H.numel()
    off = (n - nu) // 2
    y = torch.zeros((x.shape[0], n), device=DEV, dtype=torch.float64)
    if pad:
        y[:, :off] = x[:, :pad].mean(1, keepdim=True)
        y[:, off + nu:] = x[:, nu - pad:].mean(1, keepdim=True)
    y[:, off:off + nu] = x
    f = torch.fft.fft(y)
    f *= H.double()
    return torch.fft.ifft(f).real[:, off:off + nu]


def _march64(p, vol, views, step, zero_outside):
    """Ray sums of the trilinear volume, (len(views), nv, nu)."""
    f64 = dict(device=DEV, dtype=torch.float64)
    cx, cy, cz = (p.nx - 1) / 2, (p.ny - 1) / 2, (p.nz - 1) / 2
    step = step or min(p.dx, p.dy, p.dz)
    pad = torch.zeros((p.nz + 2, p.ny + 2, p.nx + 2), **f64)
    pad[1:-1, 1:-1, 1:-1] = vol
    flat = pad.reshape(-1) if zero_outside else vol.double().reshape(-1)
    out = torch.zeros((len(views), p.nv, p.nu), **f64)
    um = (torch.arange(p.nu, **f64) - (p.nu - 1) / 2)[None, :] * p.du
    vm = ((p.nv - 1) / 2 - torch.arange(p.nv, **f64))[:, None] * p.dv
    for k, s in enumerate(views):
        a = -_theta(p)[s]
        sn, cs, det = math.sin(a), math.cos(a), p.sid - p.sod
        o = (p.sod * sn, -p.sod * cs, 0.0)
        d = [um * cs - det * sn - o[0] + 0 * vm, um * sn + det * cs - o[1] + 0 * vm, vm + 0 * um]
        nrm = torch.rsqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
        d = [e * nrm for e in d]
        tn, tf = torch.full_like(nrm, -1e300), torch.full_like(nrm, 1e300)
        for e, oo, b in zip(d, o, (cx * p.dx, cy * p.dy, cz * p.dz)):
            t0, t1 = (-b - oo) / e, (b - oo) / e
            tn, tf = torch.maximum(tn, torch.minimum(t0, t1)), torch.minimum(tf, torch.maximum(t0, t1))
        length = torch.where(tf > tn, tf - tn, torch.full_like(tf, -1.0))
        og = (o[0] / p.dx + cx, cy - o[1] / p.dy, cz - o[2] / p.dz)
        dg = (d[0] / p.dx, -d[1] / p.dy, -d[2] / p.dz)
        top = float(length.max())
        acc = torch.zeros_like(nrm)
        for q in range(int(top / step) + 1 if top >= 0 else 0):
            t = tn + q * step
            idx, fr = [], []
            for oo, e, n in zip(og, dg, (p.nx, p.ny, p.nz)):
                g = oo + e * t
                i = torch.trunc(g)
                fr.append(g - i)
                lim = (-1, n) if zero_outside else (0, n - 1)
                lo, hi = i.clamp(*lim).long(), (i + 1).clamp(*lim).long()
                idx.append((lo + 1, hi + 1) if zero_outside else (lo, hi))
            nx, ny = (p.nx + 2, p.ny + 2) if zero_outside else (p.nx, p.ny)
            val = 0.0
            for zi in (0, 1):
                for yi in (0, 1):
                    base = (idx[2][zi] * ny + idx[1][yi]) * nx
                    r = flat[base + idx[0][0]] * (1 - fr[0]) + flat[base + idx[0][1]] * fr[0]
                    val = val + r * (fr[1] if yi else 1 - fr[1]) * (fr[2] if zi else 1 - fr[2])
            inside = (q * step <= length) if zero_outside else (q * step < length)
            acc += torch.where(inside, val, torch.zeros_like(val))
        out[k] = acc * step
    return out


def _shifted(x, tap):
    """x[n][z + dz][y + dy][x + dx] with zeros outside, tap = 9 (dz+1) + 3 (dy+1) + dx + 1."""
    dz, dy, dx = tap // 9 - 1, tap // 3 % 3 - 1, tap % 3 - 1
    out = torch.zeros_like(x)
    _, D, H, W, _ = x.shape
    a = [slice(max(0, -e), n - max(0, e)) for e, n in ((dz, D), (dy, H), (dx, W))]
    b = [slice(max(0, e), n - max(0, -e)) for e, n in ((dz, D), (dy, H), (dx, W))]
    out[:, a[0], a[1], a[2]] = x[:, b[0], b[1], b[2]]
    return out


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "fdk":
        p = _para(c)
        g = _gen(seed)
        raw = _line_integrals(p, _spheres(p, g), 0.5, g)
        um = (torch.arange(p.nu, device=DEV, dtype=torch.float64) - (p.nu - 1) / 2) * p.du
        vm = (torch.arange(p.nv, device=DEV, dtype=torch.float64) - (p.nv - 1) / 2) * p.dv
        af = 0.5 / p.du * (2 * math.pi / p.nproj) / 2 * (p.sid / p.sod)
        cos = p.sid * torch.rsqrt(um[None] ** 2 + vm[:, None] ** 2 + p.sid ** 2) * p.sod ** 2 * af
        n = 1 << int(p.nu).bit_length()
        f = torch.arange(n, device=DEV, dtype=torch.float64)
        f = torch.minimum(f, n - f)
        H = 2 * f / n * 0.5 * (1 + torch.cos(2 * math.pi * f / n))
        return _back64(lambda q: _filter64(raw[q], cos, H, 4).t().contiguous(), _mats64(p),
                       range(p.nx), range(p.ny), range(p.nz))
    if k == "bp":
        p, views, so = _bp_inputs(c, seed)
        t, b = _boxes(c)

        def view(q):
            v = views[q].double()
            if so is not None:
                v = v * float(so[q, 0]) + float(so[q, 1])
            return v if c["transpose"] else v.t().contiguous()
        zs = list(range(t[2], t[2] + t[5])) + list(range(b[2], b[2] + b[5]))
        return _back64(view, _mats64(p), range(t[0], t[0] + t[3]), range(t[1], t[1] + t[4]), zs)
    if k == "ratio":
        p = _para(c)
        g = _gen(seed)
        proj = _line_integrals(p, _spheres(p, g), 0.0, g).double()
        mask = torch.zeros((p.nv, p.nu), device=DEV, dtype=torch.float64)
        mask[2:-2, 2:-2] = 1
        xyz = (range(p.nx), range(p.ny), range(p.nz))
        m = _mats64(p)
        norm = _back64(lambda q: mask.t().contiguous(), m, *xyz)
        fp = _march64(p, torch.ones_like(norm), range(p.nproj), 0.0, True)
        r = torch.where(fp != 0, proj / fp, torch.zeros_like(fp)) * mask
        upd = _back64(lambda q: r[q].t().contiguous(), m, *xyz)
        return torch.where(norm != 0, upd / norm, torch.zeros_like(norm))
    if k == "filter":
        raw, cos, H = _filter_inputs(c, seed)
        out, so = [], []
        for q in range(c["views"]):
            v = _filter64(raw[q], cos, H, c["pad"])
            if c["dtype"] != "f32":
                lo, hi = float(v.min()), float(v.max())
                v = (v - lo) / (hi - lo)
                so.append((hi - lo, lo))
            out.append(v.t().contiguous() if c["transpose"] else v)
        out = torch.stack(out)
        return {"views": out} if c["dtype"] == "f32" else {"views": out, "so": np.array(so)}
    if k == "fp":
        p = _para(c)
        return _march64(p, _volume(p, _gen(seed)), range(c["views"]), c["step"], c["mode"] == 1)
    if k == "rtk":
        p = _para(c)
        g = _gen(seed)
        views = _filtered(p, g)
        vin = 1e-5 * torch.randn((p.nz, p.ny, p.nx), generator=g, device=DEV)
        return vin.double() + _back64(lambda q: views[q].double(), _mats64(p), range(p.nx),
                                      range(p.ny), range(p.nz))
    s = (c["n"], c["d"], c["h"], c["w"])
    if k == "conv":
        x, up, w, b = _conv_inputs(c, seed)
        if up is not None:
            for a in (1, 2, 3):
                up = up.repeat_interleave(2, dim=a)
            x = torch.cat([up, x], -1)
        x, w = x.double(), w.double()
        y = torch.zeros((x.numel() // c["cin"], c["cout"]), device=DEV, dtype=torch.float64)
        for t in range(27):
            y.addmm_(_shifted(x, t).reshape(-1, c["cin"]), w[t].t().contiguous())
        y += b.double()
        return y.relu_().reshape(s + (c["cout"],))
    x, y, dy, w = _bwd_inputs(c, seed)
    x, w = x.double(), w.double()
    dz = torch.where(y > 0, dy, torch.zeros_like(dy)).double()
    gw = torch.empty((27, c["cout"], c["cin"]), device=DEV, dtype=torch.float64)
    dx = torch.zeros((x.numel() // c["cin"], c["cin"]), device=DEV, dtype=torch.float64)
    flat = dz.reshape(-1, c["cout"])
    for t in range(27):
        gw[t] = flat.t().contiguous() @ _shifted(x, t).reshape(-1, c["cin"])
        dx.addmm_(_shifted(dz, 26 - t).reshape(-1, c["cout"]), w[t])
    return {"dx": dx.reshape(x.shape), "gw": gw, "gb": flat.sum(0)}

"""Performance cases: what a user of this package has it do, over the range of sizes in use.

Every case goes through the public PyTorch operators (functional.py, recon.py, ragged.py) on
tensors that are on the GPU, as a program that reconstructs, trains or iterates calls them.

  fan_fbp     fan weighting + ramp filter + fan backprojection: reconstruction of a fan scan,
              from one preview slice to a stack of 1024 x 1024 slices, in float32 and (as the
              FP64 numpy front end of the package uses it) in float64
  fan_train   the same chain as a differentiable layer: the image and the sinogram's gradient
  par_fbp     parallel projection, ramp filter, parallel backprojection of a phantom
  par_lsq     one gradient of 0.5 |FP x - y|^2, the step of an iterative reconstruction
  dd_step     distance-driven projection and the gradient defined for it
  ragged      many fan problems of different sizes with irregular angles, one launch
  fan_filter  weighting + ramp filter alone, long detector rows

Inputs are analytic sinograms of random ellipse phantoms with Poisson noise, and the phantoms
themselves; they depend on the case and the seed alone.
"""
import math

import numpy as np
import torch

from ct_recon_extensions_amd import functional as F
from ct_recon_extensions_amd import ragged, recon

DSD, DSO = 1085.6, 595.0  # source to detector and to the rotation centre, mm
HALF_FAN = 0.4407         # half the fan angle the detector covers: 736 channels of 1.30 mm
FOV = 358.4               # side of the largest image the fan covers: 512 pixels of 0.7 mm


def listed():
    return [
        # one small slice: an interactive preview, where latency and launches count
        {"name": "fan_fbp_preview", "kind": "fan_fbp", "n": 1, "ny": 256, "nx": 256, "na": 360,
         "ns": 367, "zoom": 1.0, "offset_s": 0.25, "f64": False},
        # a few slices of a zoomed, non-square region with odd sizes
        {"name": "fan_fbp_region", "kind": "fan_fbp", "n": 5, "ny": 387, "nx": 451, "na": 615,
         "ns": 561, "zoom": 0.7, "offset_s": 0.25, "f64": False},
        # a 16-slice clinical scan: the workload of the benchmark
        {"name": "fan_fbp_scan", "kind": "fan_fbp", "n": 16, "ny": 512, "nx": 512, "na": 720,
         "ns": 736, "zoom": 1.0, "offset_s": 0.0, "f64": False},
        # high-resolution slices from a 1472-channel detector
        {"name": "fan_fbp_fine", "kind": "fan_fbp", "n": 8, "ny": 1024, "nx": 1024, "na": 1440,
         "ns": 1472, "zoom": 1.0, "offset_s": 0.25, "f64": False},
        # FP64, as the numpy front end and reference runs compute
        {"name": "fan_fbp_double", "kind": "fan_fbp", "n": 2, "ny": 512, "nx": 512, "na": 720,
         "ns": 736, "zoom": 1.0, "offset_s": 0.0, "f64": True},
        # the filtered backprojection as a layer of a network, forward and backward
        {"name": "fan_train_batch", "kind": "fan_train", "n": 4, "ny": 512, "nx": 512, "na": 720,
         "ns": 736, "zoom": 1.0, "offset_s": 0.0, "f64": False},
        # a parallel scan simulated and reconstructed: the smallest end-to-end chain
        {"name": "par_fbp_phantom", "kind": "par_fbp", "n": 1, "ny": 256, "nx": 256, "na": 360,
         "ns": 367},
        # one step of an iterative reconstruction of eight slices
        {"name": "par_lsq_batch", "kind": "par_lsq", "n": 8, "side": 512, "na": 720, "ns": 729},
        # the same for one slice of a small scan with odd sizes
        {"name": "par_lsq_slice", "kind": "par_lsq", "n": 1, "side": 333, "na": 415, "ns": 475},
        # distance-driven projector pair, as in a model-based reconstruction
        {"name": "dd_step_batch", "kind": "dd_step", "n": 8, "ny": 512, "nx": 512, "na": 720,
         "ns": 729},
        # a batch of unrelated scans with jittered view angles
        {"name": "ragged_batch", "kind": "ragged", "count": 64, "most": 512, "problems": 20261204},
        # filter of a whole high-resolution scan
        {"name": "fan_filter_long", "kind": "fan_filter", "n": 32, "na": 1440, "ns": 1472,
         "offset_s": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fan_fbp", "fan_fbp", "fan_fbp", "fan_train", "par_fbp", "par_lsq",
                       "par_lsq", "dd_step", "ragged", "fan_filter"])
    if kind == "ragged":
        return {"kind": kind, "count": _log(rng, 4, 64), "most": rng.choice([256, 384, 512]),
                "problems": rng.randrange(1 << 30)}
    if kind == "fan_filter":
        return {"kind": kind, "n": _log(rng, 1, 32), "na": _log(rng, 180, 1440),
                "ns": _log(rng, 256, 1472), "offset_s": rng.choice([0.0, 0.25])}
    side = _log(rng, 192, 1024)
    na, ns = int(side * rng.uniform(1.0, 1.6)), int(side * rng.uniform(1.3, 1.6))
    if kind == "par_lsq":
        side = min(side, 640)
        na, ns = min(na, 900), min(max(ns, side), 960)
        return {"kind": kind, "n": min(_log(rng, 1, 8), max(1, int(8 * (512 / side) ** 3))),
                "side": side, "na": na, "ns": ns}
    if kind in ("par_fbp", "dd_step"):
        side = min(side, 512)
        na, ns = min(na, 720), min(ns, 736)
        c = {"kind": kind, "n": _log(rng, 1, 8), "ny": max(160, side - rng.randrange(64)),
             "nx": side, "na": na, "ns": ns}
        return c
    c = {"kind": kind, "n": 1, "ny": max(160, side - rng.choice([0, 0, rng.randrange(64)])),
         "nx": side, "na": na, "ns": min(ns, 1472),
         "zoom": rng.choice([1.0, 1.0, rng.uniform(0.5, 1.0)]),
         "offset_s": rng.choice([0.0, 0.25]), "f64": kind == "fan_fbp" and rng.random() < 0.2}
    # as many slices as the largest listed case has work for, 32 at most
    views = c["ny"] * c["nx"] * c["na"]
    most = (4e8 if c["f64"] else 2e9 if kind == "fan_train" else 1.1e10) / views
    c["n"] = _log(rng, 1, max(1, min(32, int(most))))
    if c["f64"] and views > 4e8:
        c["f64"] = False
    return c


# ------------------------------------------------------------------ geometry
def _fan_kw(c):
    return {"img_shape": [c["ny"], c["nx"]],
            "img_space": [_pixel(c), _pixel(c)],
            "proj_shape": [c["na"], c["ns"]], "channel_space": _pitch(c["ns"]),
            "channel_offset": c["offset_s"], "orbit": 2 * math.pi / c["na"], "dso": DSO,
            "dsd": DSD}


def _pixel(c):
    return FOV * c["zoom"] / max(c["ny"], c["nx"])


def _pitch(ns):
    return 2 * HALF_FAN * DSD / ns


def _filter_kw(c):
    return {"proj_shape": [c["na"], c["ns"]], "channel_space": _pitch(c["ns"]),
            "channel_offset": c["offset_s"], "dso": DSO, "dsd": DSD, "tp": "fan"}


def _par_kw(c):
    # pixels and channels of pitch 1, 180 degrees
    return {"img_shape": [c["ny"], c["nx"]], "img_space": [1.0, 1.0],
            "proj_shape": [c["na"], c["ns"]], "channel_space": 1.0,
            "orbit": math.pi / c["na"]}


def _scan(c):
    return recon.ParallelScan(n=c["side"], na=c["na"], ns=c["ns"])


# -------------------------------------------------------------------- inputs
def _ellipses(rs, radius):
    """A body and eleven features in it: x0, y0, a, b, phi, density (1/mm)."""
    e = np.empty((12, 6))
    e[0] = (0, 0, 0.92 * radius, rs.uniform(0.6, 0.9) * radius, rs.uniform(0, math.pi), 0.02)
    r, t = 0.5 * radius * np.sqrt(rs.uniform(size=11)), rs.uniform(0, 2 * math.pi, 11)
    e[1:, 0], e[1:, 1] = r * np.cos(t), r * np.sin(t)
    e[1:, 2:4] = rs.uniform(0.02, 0.3, (11, 2)) * radius
    e[1:, 4] = rs.uniform(0, math.pi, 11)
    e[1:, 5] = rs.uniform(-0.008, 0.01, 11)
    return e


def _line_integrals(ell, theta, t):
    """Integrals along the rays x cos(theta) + y sin(theta) = t (FP64 tensors)."""
    c, s = torch.cos(theta), torch.sin(theta)
    out = torch.zeros(torch.broadcast_shapes(theta.shape, t.shape), dtype=torch.float64,
                      device=t.device)
    for x0, y0, a, b, phi, rho in ell:
        m2 = (a * torch.cos(theta - phi)) ** 2 + (b * torch.sin(theta - phi)) ** 2
        q = (m2 - (t - x0 * c - y0 * s) ** 2).clamp_min_(0.0)
        out += 2.0 * rho * a * b * q.sqrt_() / m2
    return out


def _noisy(p, rs, gen, dtype):
    """Counts of 10^4 to 10^6 photons a ray, back to line integrals."""
    i0 = 10.0 ** rs.uniform(4, 6)
    counts = torch.poisson(i0 * torch.exp(-p), generator=gen)
    return (-torch.log(counts.clamp_min_(1.0) / i0)).to(dtype)


def _fan_sinogram(c, beta, ds, dso, radius, n, rs, gen, dtype):
    na, ns = len(beta), c["ns"]
    gamma = (torch.arange(ns, dtype=torch.float64, device="cuda")
             - ((ns - 1) / 2 + c["offset_s"])) * (ds / DSD)
    theta = torch.as_tensor(beta, device="cuda")[:, None] + gamma[None, :]
    t = (dso * torch.sin(gamma))[None, :]
    out = torch.empty((n, na, ns), dtype=dtype, device="cuda")
    for b in range(n):
        out[b] = _noisy(_line_integrals(_ellipses(rs, radius), theta, t), rs, gen, dtype)
    return out


def _image(ell, ny, nx, scale):
    y = ((ny - 1) / 2 - torch.arange(ny, dtype=torch.float64, device="cuda"))[:, None]
    x = (torch.arange(nx, dtype=torch.float64, device="cuda") - (nx - 1) / 2)[None, :]
    img = torch.zeros((ny, nx), dtype=torch.float64, device="cuda")
    for x0, y0, a, b, phi, rho in ell:
        cp, sp = math.cos(phi), math.sin(phi)
        u, v = (x - x0) * cp + (y - y0) * sp, (y - y0) * cp - (x - x0) * sp
        img += scale * rho * ((u / a) ** 2 + (v / b) ** 2 <= 1.0)
    return img


def _images(n, ny, nx, rs, scale=1.0):
    ells = [_ellipses(rs, 0.5 * min(ny, nx)) for _ in range(n)]
    return torch.stack([_image(e, ny, nx, scale) for e in ells]).float(), ells


def _inputs(c, seed):
    """What the case's call is given, as a dict of tensors (and the ragged batch's geometry)."""
    rs = np.random.RandomState(seed % (1 << 32))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = c["kind"]
    if kind in ("fan_fbp", "fan_train", "fan_filter"):
        dtype = torch.float64 if c.get("f64") else torch.float32
        beta = 2 * math.pi / c["na"] * np.arange(c["na"])
        d = {"proj": _fan_sinogram(c, beta, _pitch(c["ns"]), DSO, 0.5 * FOV, c["n"], rs, gen,
                                   dtype)}
        if kind == "fan_train":  # the loss' gradient: the noise and edges of an image
            g, _ = _images(c["n"], c["ny"], c["nx"], rs)
            d["grad"] = g + 0.002 * torch.randn(g.shape, generator=gen, device="cuda")
        return d
    if kind in ("par_fbp", "dd_step"):
        img, _ = _images(c["n"], c["ny"], c["nx"], rs)
        if kind == "par_fbp":
            return {"img": img}
        return {"img": img, "grad": torch.randn((c["n"], c["na"], c["ns"]), generator=gen,
                                                device="cuda")}
    if kind == "par_lsq":  # an early iterate (the phantom at 0.6) and the measured sinogram
        img, ells = _images(c["n"], c["side"], c["side"], rs, 0.6)
        th = (math.pi / c["na"] * torch.arange(c["na"], dtype=torch.float64, device="cuda"))
        t = (torch.arange(c["ns"], dtype=torch.float64, device="cuda") - (c["ns"] - 1) / 2)
        y = [_noisy(_line_integrals(e, th[:, None], t[None, :]), rs, gen, torch.float32)
             for e in ells]
        return {"img": img, "y": torch.stack(y)}
    sizes = [s for s in (128, 256, 384, 512) if s <= c["most"]]
    params, angles = ragged.random_fan_problems(c["count"], c["problems"], sizes=sizes)
    projs = [_fan_sinogram({"ns": p.ns, "offset_s": p.offset_s}, a, p.ds, p.dso,
                           0.45 * p.nx * p.dx, 1, rs, gen, torch.float32)[0]
             for p, a in zip(params, angles)]
    return {"params": params, "angles": angles, "projs": projs}


# ----------------------------------------------------------------- the calls
def prepare(case, seed):
    s = {"case": case, **_inputs(case, seed)}
    kind = case["kind"]
    if kind in ("fan_fbp", "fan_train"):
        s["filter"], s["bp"] = _filter_kw(case), _fan_kw(case)
    elif kind == "fan_filter":
        s["filter"] = _filter_kw(case)
    elif kind in ("par_fbp", "dd_step"):
        s["kw"] = _par_kw(case)
    elif kind == "par_lsq":
        s["fp"], _ = recon.projector(_scan(case))
    else:
        # a plan as a program makes it that does not tune every batch it meets
        plan = ragged.RaggedFanBackprojection2DAngle(s.pop("params"), s.pop("angles"),
                                                     autotune=False, tile=0, vchunk=16)
        for dst, src in zip(plan.projs, s.pop("projs")):
            dst.copy_(src)
        s["plan"] = plan
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind == "fan_fbp":
        return F.fan_backprojection_2d(F.fan_filter(state["proj"], **state["filter"]),
                                       **state["bp"])
    if kind == "fan_train":
        x = state["proj"].detach().requires_grad_(True)
        img = F.fan_backprojection_2d(F.fan_filter(x, **state["filter"]), **state["bp"])
        (g,) = torch.autograd.grad(img, x, state["grad"])
        return img.detach(), g
    if kind == "fan_filter":
        return F.fan_filter(state["proj"], **state["filter"])
    if kind == "par_fbp":
        kw, c = state["kw"], state["case"]
        p = F.parallel_projection_2d(state["img"], **kw)
        return p, F.parallel_backprojection_2d(F.ramp_filter(p, c["ns"], c["na"], 1.0), **kw)
    if kind == "par_lsq":
        return recon.loss_and_grad(state["img"], state["y"], state["fp"])
    if kind == "dd_step":
        x = state["img"].detach().requires_grad_(True)
        p = F.parallel_projection_2d(x, method="disdriven", **state["kw"])
        (g,) = torch.autograd.grad(p, x, state["grad"])
        return p.detach(), g
    state["plan"]()
    return state["plan"].img_flat


# ------------------------------------------------------ what cannot be spared
def _filter_work(rows, ns, item):
    # in and out once; two real transforms of the zero-padded row
    length = 1 << (2 * ns - 1).bit_length()
    return 2 * rows * ns * item, rows * 5.0 * length * math.log2(length)


def work(case):
    c, kind = case, case["kind"]
    if kind == "ragged":
        params, _ = ragged.random_fan_problems(
            c["count"], c["problems"], sizes=[s for s in (128, 256, 384, 512) if s <= c["most"]])
        return {"bytes": 4.0 * sum(p.na * p.ns + p.nx * p.ny for p in params),
                "flops": 16.0 * sum(p.na * p.nx * p.ny for p in params)}
    item = 8 if c.get("f64") else 4
    sino = c["na"] * c["ns"] * c["n"]
    if kind == "fan_filter":
        by, fl = _filter_work(c["n"] * c["na"], c["ns"], item)
        return {"bytes": float(by), "flops": fl}
    ny, nx = (c["side"], c["side"]) if "side" in c else (c["ny"], c["nx"])
    img, pv = ny * nx * c["n"], ny * nx * c["na"]
    # per pixel and view: its detector position and weight once (12), then two
    # multiply-adds for every slice
    bp = pv * (12.0 + 4.0 * c["n"])
    rays = c["na"] * c["ns"] * max(ny, nx) * (4.0 + 4.0 * c["n"])
    _, fl = _filter_work(c["n"] * c["na"], c["ns"], item)
    if kind == "fan_fbp":
        return {"bytes": float(item * (sino + img)), "flops": fl + bp}
    if kind == "fan_train":
        return {"bytes": 4.0 * (2 * sino + 2 * img), "flops": 2 * (fl + bp)}
    if kind == "par_fbp":
        return {"bytes": 4.0 * (sino + 2 * img), "flops": rays + fl + bp}
    if kind == "par_lsq":
        return {"bytes": 4.0 * (sino + 2 * img), "flops": rays + bp}
    return {"bytes": 4.0 * (2 * sino + 2 * img), "flops": 1.5 * (rays + bp)}


# ------------------------------------------------------------ 64-bit results
def _cells(n, space, sign):
    """Pixel centres, accumulated from the first one."""
    step = np.full(n, sign * space)
    step[0] = -sign * (n - 1) / 2.0 * space
    return torch.from_numpy(np.cumsum(step)).cuda()


def _angles(na, orbit):
    step = np.full(na, orbit)
    step[0] = 0.0
    return np.cumsum(step)


def _fan_filter64(proj, ns, offset_s, fan=True, weight=True):
    ds = _pitch(ns) if fan else 1.0
    m = np.arange(-(ns - 1), ns)
    h = np.zeros(2 * ns - 1)
    odd = m % 2 != 0
    h[odd] = (-1.0 / (math.pi * DSD * np.sin(m[odd] * ds / DSD)) ** 2 if fan
              else -1.0 / (math.pi * ds * m[odd]) ** 2)
    h[ns - 1] = 0.25 / ds ** 2
    i = np.arange(ns)
    toeplitz = torch.from_numpy(ds * h[i[:, None] - i[None, :] + ns - 1]).cuda()
    w = _cos64(ns, ds, offset_s) if weight else 1.0
    return ((proj.double() * w).reshape(-1, ns) @ toeplitz).reshape(proj.shape)


def _cos64(ns, ds, offset_s):
    s = (torch.arange(ns, dtype=torch.float64, device="cuda") - ((ns - 1) / 2 + offset_s)) * ds
    return DSO / DSD * torch.cos(s / DSD).abs()


def _fan_taps(c, ds, dso, px, py, k, beta):
    """Left tap, fraction and weight of every pixel of one fan view (0 off the detector)."""
    sb, cb = math.sin(beta), math.cos(beta)
    x, y = px[None, :], py[:, None]
    d, r = dso + x * sb - y * cb, x * cb + y * sb
    return _taps(torch.atan2(r, d) * DSD / ds + k, DSD * DSD / (d * d + r * r), c["ns"])


def _taps(s, w, ns):
    w = torch.where((s >= 0) & (s <= ns - 1), w, 0.0)
    i = s.floor().clamp(0, ns - 2)
    return i.long().reshape(-1), (s - i).reshape(-1), w.reshape(-1)


def _gather(row, taps):
    i, u, w = taps
    return w * ((1 - u) * row[:, i] + u * row[:, i + 1])


def _fan_bp64(c, proj, beta, ds, dso, dx, scale, ny, nx):
    px, py = _cells(nx, dx, 1.0), _cells(ny, dx, -1.0)
    k = (c["ns"] - 1) / 2 + c["offset_s"]
    out = torch.zeros((proj.shape[0], ny * nx), dtype=torch.float64, device="cuda")
    for v, b in enumerate(beta):
        out += _gather(proj[:, v], _fan_taps(c, ds, dso, px, py, k, float(b)))
    return (scale * out).reshape(-1, ny, nx)


def _fan_bpt64(c, img, beta, ds, dso, dx, scale, ny, nx):
    px, py = _cells(nx, dx, 1.0), _cells(ny, dx, -1.0)
    k = (c["ns"] - 1) / 2 + c["offset_s"]
    flat = img.reshape(img.shape[0], -1)
    out = torch.zeros((img.shape[0], len(beta), c["ns"]), dtype=torch.float64, device="cuda")
    for v, b in enumerate(beta):
        i, u, w = _fan_taps(c, ds, dso, px, py, k, float(b))
        out[:, v].index_add_(1, i, flat * (w * (1 - u)))
        out[:, v].index_add_(1, i + 1, flat * (w * u))
    return scale * out


def _branch(ang):
    q = math.pi / 4
    return not (q <= ang < 3 * q or 5 * q <= ang < 7 * q)


def _rays(c, ny, nx):
    """Per view: x-branch?, start of every channel, step per row, factor, half a channel."""
    cx, cy, cs = (nx - 1) / 2, (ny - 1) / 2, (c["ns"] - 1) / 2
    for ang in _angles(c["na"], math.pi / c["na"]):
        sa, ca = math.sin(ang), math.cos(ang)
        if _branch(ang):
            step, ch, dw = sa / ca, 1.0 / ca, abs(1.0 / ca)
            begin = cx - cy * step - cs * ch
        else:
            step, ch, dw = ca / sa, -1.0 / sa, abs(1.0 / sa)
            begin = cy - cx * step - cs * ch
        start = np.full(c["ns"], ch)
        start[0] = begin
        yield _branch(ang), np.cumsum(start), step, dw, ch / 2


def _fp64(c, img, ny, nx, driven):
    """Ray-driven (driven = 1) or distance-driven (2) parallel projection."""
    img = img.double()
    rays = list(_rays(c, ny, nx))
    out = torch.zeros((img.shape[0], c["na"], c["ns"]), dtype=torch.float64, device="cuda")
    for xb in (True, False):
        views = [v for v, r in enumerate(rays) if r[0] == xb]
        if not views:
            continue
        pos, step, dw, half = (torch.as_tensor(np.array([rays[v][k] for v in views]),
                                               device="cuda") for k in (1, 2, 3, 4))
        step, dw, half = step[:, None], dw[:, None], half[:, None].abs()
        rows = img if xb else img.transpose(1, 2).contiguous()
        hi = rows.shape[2] - 1
        total = torch.zeros((img.shape[0],) + pos.shape, dtype=torch.float64, device="cuda")
        left, right = pos - half, pos + half
        for k in range(rows.shape[1]):
            row = rows[:, k]
            if driven == 1:
                on = ((pos >= 0) & (pos <= hi)).double()
                i = pos.floor().clamp(0, hi - 1)
                u = pos - i
                i = i.long()
                total += on * ((1 - u) * row[:, i] + u * row[:, i + 1])
                pos += step
                continue
            fl, tsum, lsum = left.floor(), 0.0, 0.0
            for m in range(int(2 * float(half.max())) + 2):
                v = fl + m
                ok = (fl >= 0) & (v < right.ceil()) & (v < hi)
                ln = torch.where(ok, torch.minimum(v + 1, right) - torch.maximum(v, left), 0.0)
                i = v.clamp(0, hi - 1).long()
                tsum = tsum + ln * (row[:, i] + row[:, i + 1]) / 2
                lsum = lsum + ln
            total += torch.where(lsum > 0, tsum / lsum, 0.0)
            left += step
            right += step
        out[:, views] = total * dw
    return out


def _fpt64(c, proj, ny, nx, driven):
    """Gradient of _fp64, per pixel: the channels its footprint on the detector meets."""
    cx, cy, cs, ns = (nx - 1) / 2, (ny - 1) / 2, (c["ns"] - 1) / 2, c["ns"]
    proj = proj.double()
    out = torch.zeros((proj.shape[0], ny, nx), dtype=torch.float64, device="cuda")
    for v, ang in enumerate(_angles(c["na"], math.pi / c["na"])):
        sa, ca = math.sin(ang), math.cos(ang)
        xb = _branch(ang)
        o1, o2, w = (ca, -sa, abs(1.0 / ca)) if xb else (-sa, ca, abs(1.0 / sa))
        begin = cs - (cx if xb else cy) * o1 - (cy if xb else cx) * o2
        start = np.full(ny if xb else nx, o2)
        start[0] = begin
        n = nx if xb else ny
        along = torch.arange(n, dtype=torch.float64, device="cuda")
        mid = torch.from_numpy(np.cumsum(start)).cuda()[:, None] + (along * o1)[None, :]
        one, two = mid - o1, mid + o1
        one[:, 0], two[:, -1] = mid[:, 0], mid[:, -1]
        left, right = torch.minimum(one, two), torch.maximum(one, two)
        first = left.ceil() if driven == 1 else (left - 0.5).ceil()
        last = right.floor() if driven == 1 else (right + 0.5).floor()
        acc = 0.0
        for m in range(int(2 * abs(o1)) + (2 if driven == 1 else 3)):
            ch = first + m
            ok = (ch >= 0) & (ch <= last) & (ch < ns)
            if driven == 1:
                wt = 1.0 - ((mid - ch) / o1).abs()
            else:
                ok &= first >= 0
                wt = (torch.minimum(ch + 0.5, right) - torch.maximum(ch - 0.5, left)) / 2
            acc = acc + torch.where(ok, wt, 0.0) * proj[:, v][:, ch.clamp(0, ns - 1).long()]
        out += w * (acc if xb else acc.transpose(1, 2))
    return out


def _par_bp64(c, proj, ny, nx):
    px, py = _cells(nx, 1.0, 1.0), _cells(ny, 1.0, -1.0)
    out = torch.zeros((proj.shape[0], ny * nx), dtype=torch.float64, device="cuda")
    for v, ang in enumerate(_angles(c["na"], math.pi / c["na"])):
        s = (px * math.cos(ang))[None, :] + (py * math.sin(ang))[:, None] + (c["ns"] - 1) / 2
        out += _gather(proj[:, v], _taps(s, torch.ones_like(s), c["ns"]))
    return (math.pi / c["na"] * out).reshape(-1, ny, nx)


def exact(case, seed):
    c, kind, d = case, case["kind"], _inputs(case, seed)
    if kind == "fan_filter":
        return _fan_filter64(d["proj"], c["ns"], c["offset_s"])
    if kind in ("fan_fbp", "fan_train"):
        args = (_angles(c["na"], 2 * math.pi / c["na"]), _pitch(c["ns"]), DSO, _pixel(c),
                math.pi / c["na"], c["ny"], c["nx"])
        img = _fan_bp64(c, _fan_filter64(d["proj"], c["ns"], c["offset_s"]), *args)
        if kind == "fan_fbp":
            return img
        g = _fan_filter64(_fan_bpt64(c, d["grad"].double(), *args), c["ns"], 0.0, weight=False)
        return img, g * _cos64(c["ns"], _pitch(c["ns"]), c["offset_s"])
    if kind == "par_fbp":
        p = _fp64(c, d["img"], c["ny"], c["nx"], 1)
        return p, _par_bp64(c, _fan_filter64(p, c["ns"], 0.0, fan=False, weight=False),
                            c["ny"], c["nx"])
    if kind == "par_lsq":
        r = _fp64(c, d["img"], c["side"], c["side"], 1) - d["y"].double()
        return 0.5 * (r * r).sum(), _fpt64(c, r, c["side"], c["side"], 1)
    if kind == "dd_step":
        return (_fp64(c, d["img"], c["ny"], c["nx"], 2),
                _fpt64(c, d["grad"], c["ny"], c["nx"], 2))
    out = []
    for p, a, proj in zip(d["params"], d["angles"], d["projs"]):
        g = {"ns": p.ns, "offset_s": p.offset_s}
        out.append(_fan_bp64(g, proj[None].double(), a, p.ds, p.dso, p.dx, 1.0, p.ny, p.nx))
    return torch.cat([o.reshape(-1) for o in out])

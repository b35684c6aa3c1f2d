"""Performance cases of the snapshot imager: what is timed, on which inputs, and the exact results.

A case images synthetic snapshots of a station array through one of the package's public calls:

* ``single``:  ``image_snapshot``, one device-resident snapshot, the ordinary call;
* ``planned``: ``image_snapshot(plan=...)``, new visibilities on a geometry already planned;
* ``pair``:    ``preprocess_measurement_set_gpu`` then ``FIpipeDevice``, the two-step form;
* ``batch``:   ``image_snapshot_batch(wait=False)``, consecutive snapshots of one size;
* ``mixed``:   ``image_snapshot_batch`` over snapshots of several image sizes and hour angles;
* ``host``:    ``fipipe_host``, preprocessed samples in host memory, archive semantics.

The array's stations belong to the case (a telescope does not move); the sky, the noise, the
flags, the weights and a few seconds of hour angle come from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import svdimager_amd as S
from svdimager_amd import imager

C_LIGHT = 299792458.0
LATITUDE = math.radians(-26.82)
DECLINATION = math.radians(-30.0)
ARRAY_CENTER_X = -2565018.0
NUM_SOURCES = 50
BETA = 15.3704324328
CONV_NORM = 2.4937047051153827
TARGET_ERROR = 1e-2
TARGET_ALPHA = 10.0
EXACT_LIMIT = 1.3e10         # footprint cells x values per cell that exact() sums, at most
MIXED_SIZES = (1024, 2048, 512, 1024, 512, 2048, 1024, 512)

# A station array, a band and an image; every case overrides what differs.
_BASE = dict(call="single", stations=512, disk=False, radius=35000.0, channels=64, f_lo=50e6, f_hi=350e6,
             size=1024, cell=2e-5, ha=0.0, flagged=0.1, removed=0.0, weights=True, signed=False, count=1)


def _case(name, **over):
    return dict(_BASE, name=name, **over) if name else dict(_BASE, **over)


def listed():
    return [
        # A 64-station test array: the smallest call, bound by launches and the host.
        _case("small-128", stations=64, disk=True, radius=1000.0, channels=16, f_lo=100e6, f_hi=150e6, size=128,
              cell=1e-4, flagged=0.05),
        # An odd image size from an odd number of channels without WEIGHT_SPECTRUM, as a user who
        # does not think of FFT lengths asks for it; the signed image.
        _case("odd-301", stations=100, disk=True, radius=3000.0, channels=31, f_lo=100e6, f_hi=160e6, size=301,
              cell=5e-5, flagged=0.05, weights=False, signed=True),
        # A mid-size array after flagged rows were dropped (a row count that no vector width
        # divides) at a round, not power-of-two, image size.
        _case("ragged-1000", stations=256, channels=48, size=1000, ha=1.5, removed=0.1),
        # Snapshots of the serving mix: the small image off transit.
        _case("skalow-512", size=512, ha=-2.0, removed=0.38, flagged=0.0),
        # The headline snapshot: 512 stations, 64 channels, 8.4 M samples, 1024^2.
        _case("skalow-1024"),
        # The serving mix's dearest: 2048^2 far from transit, several slabs of many terms.
        _case("skalow-2048-far", size=2048, ha=4.0, removed=0.55, flagged=0.0, signed=True),
        # The precision form: 16.7 M samples at 4096^2.
        _case("skalow-4096", channels=128, size=4096),
        # Fixed geometry re-imaged with new visibilities (calibration loops).
        _case("planned-1024", call="planned", signed=True),
        # The reference's own two calls on device buffers, materialised Bin included.
        _case("pair-1024", call="pair", stations=256, ha=-1.0),
        # The archive CLI's call on host buffers, copies included.
        _case("host-512", call="host", stations=256, channels=32, size=512, flagged=0.0),
        # Production: eight consecutive snapshots in one asynchronous batched call.
        _case("batch-1024x8", call="batch", count=8),
        # The batching form: eight snapshots over +-4 h, uneven rows, three image sizes.
        _case("mixed-8", call="mixed", count=8, flagged=0.0, removed=0.3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n, most):
    for p in range(2, most + 1):
        while n % p == 0:
            n //= p
    return n == 1


def _round_size(n):
    """The nearest even size whose only prime factors are 2, 3, 5 and 7."""
    return next(m for d in range(n) for m in (n - d, n + d) if m % 2 == 0 and _smooth(m, 7))


def draw(rng):
    while True:
        call = rng.choice(("single", "single", "single", "single", "planned", "pair", "host", "batch", "mixed"))
        small = rng.random() < 0.3
        if small:
            c = _case(None, call=call, stations=_log_int(rng, 32, 160), disk=True,
                      radius=math.exp(rng.uniform(math.log(500.0), math.log(4000.0))), channels=_log_int(rng, 4, 64),
                      f_lo=100e6, f_hi=rng.uniform(130e6, 200e6))
        else:
            c = _case(None, call=call, stations=_log_int(rng, 96, 512), channels=_log_int(rng, 12, 96),
                      f_hi=rng.uniform(150e6, 350e6))
        odd = rng.random() < 0.2
        n = _log_int(rng, 96, 600) if odd or small else _log_int(rng, 256, 2200)
        c["size"] = n | 1 if odd else _round_size(n)
        c["cell"] = min(rng.uniform(5e-5, 1.2e-4) if small else rng.uniform(1.2e-5, 3e-5), 0.041 / c["size"])
        c["ha"] = rng.uniform(-4.0, 4.0)
        c["flagged"] = rng.choice((0.0, 0.05, 0.1, 0.2))
        c["removed"] = rng.choice((0.0, rng.uniform(0.0, 0.6)))
        c["weights"] = rng.random() < 0.75
        c["signed"] = rng.random() < 0.35
        c["count"] = rng.randint(2, 6) if call in ("batch", "mixed") else 1
        samples = c["count"] * _num_rows(c) * c["channels"]
        cells = direct = alpha = 0.0
        for i in range(c["count"]):
            p = _plan64(*_geometry(c, 0, i), *_image(c, i), archive=call == "host")
            G = (3 * _image(c, i)[0] + 1) // 2
            cells += p["slabs"] * p["terms"] * G * G
            direct += 0.0 if _smooth(G, 13) else 16.0 * p["slabs"] * p["terms"] * G ** 3
            alpha = max(alpha, p["alpha"])
        # (Transform lengths with a prime factor above 13 are dearer; the Bessel series of exact()
        # holds to 12.)
        if samples <= 3.2e7 and cells <= 6e8 and direct <= 1e11 and alpha <= 12.0:
            return c


# ------------------------------------------------------------------------------------- inputs

def _image(case, i):
    """Image side and cell of the case's snapshot i."""
    if case["call"] != "mixed":
        return case["size"], case["cell"]
    size = MIXED_SIZES[i % len(MIXED_SIZES)]
    return size, min(case["cell"], 0.041 / size)


def _num_rows(case, i=0):
    rows = case["stations"] * (case["stations"] - 1) // 2
    removed = case["removed"] * (0.4 + 0.3 * (i % 5)) if case["call"] == "mixed" else case["removed"]
    keep = int(round(rows * (1.0 - removed)))
    return keep | 1 if removed > 0 else keep


def _geometry(case, seed, i):
    """uvw (R, 3) in metres and the channel frequencies of the case's snapshot i, FP64."""
    rng = np.random.default_rng([case["stations"], int(case["radius"])])
    n = case["stations"]
    theta = rng.uniform(0.0, 2.0 * math.pi, n)
    u = rng.uniform(0.0, 1.0, n)
    radius = case["radius"] * np.sqrt(u) if case["disk"] else np.exp(math.log(10.0) + u * math.log(case["radius"] / 10.0))
    east, north, up = radius * np.cos(theta), radius * np.sin(theta), rng.normal(0.0, 5.0 if case["disk"] else 20.0, n)
    sl, cl = math.sin(LATITUDE), math.cos(LATITUDE)
    xyz = np.stack([-sl * north + cl * up, east, cl * north + sl * up], axis=1)
    ha = case["ha"] if case["call"] != "mixed" else -4.0 + 8.0 * i / max(1, case["count"] - 1)
    h = (ha + (10.0 * (seed % 64) + 10.0 * i) / 3600.0) * math.pi / 12.0
    a, b = np.triu_indices(n, k=1)
    x, y, z = (xyz[b] - xyz[a]).T
    sh, ch, sd, cd = math.sin(h), math.cos(h), math.sin(DECLINATION), math.cos(DECLINATION)
    uvw = np.stack([sh * x + ch * y, -sd * ch * x + sd * sh * y + cd * z, cd * ch * x - cd * sh * y + sd * z], axis=1)
    rows = _num_rows(case, i)
    if rows < uvw.shape[0]:
        uvw = uvw[np.sort(np.random.default_rng([case["stations"], i]).choice(uvw.shape[0], rows, replace=False))]
    return np.ascontiguousarray(uvw), np.linspace(case["f_lo"], case["f_hi"], case["channels"])


def _snapshot(case, seed, i, dev):
    """The case's snapshot i: the fields of a MeasurementSet snapshot, device-resident."""
    uvw, freq = _geometry(case, seed, i)
    size, cell = _image(case, i)
    gen = torch.Generator(device=dev)
    gen.manual_seed(1009 * int(seed) + i)
    rng = np.random.default_rng([int(seed), i])
    R, C = uvw.shape[0], len(freq)
    lm = rng.uniform(-0.35, 0.35, (2, NUM_SOURCES)) * size * cell
    flux = np.minimum(0.05 * rng.uniform(0.0, 1.0, NUM_SOURCES) ** (-1.0 / 1.8), 20.0)
    lmn = np.concatenate([lm, np.sqrt(1.0 - (lm ** 2).sum(0, keepdims=True)) - 1.0])
    uvw_d = torch.from_numpy(uvw).to(dev)
    delay = uvw_d @ torch.from_numpy(lmn).to(dev)
    amp = torch.from_numpy(flux.astype(np.float32)).to(dev)
    model = torch.empty((2, C, R), dtype=torch.float32, device=dev)
    for c in range(C):
        turn = delay * (freq[c] / C_LIGHT)
        ang = (turn - torch.round(turn)).float() * (-2.0 * math.pi)
        model[0, c] = torch.cos(ang) @ amp
        model[1, c] = torch.sin(ang) @ amp
    snap = {"uvw": uvw_d, "freq": torch.from_numpy(freq).to(dev), "num_rows": R, "num_channels": C,
            "array_center_x": ARRAY_CENTER_X}
    for pol in (0, 3):
        for part, name in ((0, "re"), (1, "im")):
            noise = torch.randn((C, R), generator=gen, device=dev) * 0.01
            snap[f"vis{pol}_{name}"] = (model[part] + noise).reshape(-1)
    flags = (torch.rand(R, generator=gen, device=dev) < case["flagged"]).to(torch.uint8)
    for pol in (0, 3):
        snap[f"flag{pol}"] = flags.repeat(C)
        snap[f"weight{pol}"] = torch.rand(R * C, generator=gen, device=dev) * 0.5 + 0.5 if case["weights"] else None
    return snap


_CONTEXT = []


def _context():
    """The program's one imaging context."""
    if not _CONTEXT:
        _CONTEXT.append(S.Context(0))
    return _CONTEXT[0]


def _options(case):
    return {"output": S.OUTPUT_SIGNED if case["signed"] else S.OUTPUT_DIRTY}


def _host_samples(case, seed, dev):
    """The preparation step's outputs (rotated baselines in wavelengths, rotation, collapsed
    visibilities) in FP32, from plain torch."""
    snap = _snapshot(case, seed, 0, dev)
    rot = _rotation64(snap["uvw"], snap["freq"])
    b, vis = _fold64(snap, rot)
    return b.float(), rot.float(), vis.real.float(), vis.imag.float()


def prepare(case, seed):
    dev = torch.device("cuda", 0)
    state = {"case": case, "ctx": _context()}
    if case["call"] == "host":
        b, rot, re, im = _host_samples(case, seed, dev)
        state["host"] = [t.cpu().numpy() for t in (re, im, b, rot)]
        return state
    state["snaps"] = [S.DeviceSnapshot(_snapshot(case, seed, i, dev), dev) for i in range(case["count"])]
    state["sizes"] = [_image(case, i)[0] for i in range(case["count"])]
    state["cells"] = [_image(case, i)[1] for i in range(case["count"])]
    state["images"] = [torch.empty((n, n), dtype=torch.float32, device=dev) for n in state["sizes"]]
    if case["call"] == "planned":
        _, state["plan"] = imager.image_snapshot(state["ctx"], state["snaps"][0], case["size"], case["cell"],
                                                 image=state["images"][0], **_options(case))
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    call, opts = case["call"], _options(case)
    if call == "host":
        image, plan = imager.fipipe_host(ctx, *state["host"], case["size"], case["cell"], **opts)
        return {"image": image, "terms": plan["num_terms"]}
    snaps, images = state["snaps"], state["images"]
    if call == "pair":
        pre = imager.preprocess_measurement_set_gpu(ctx, snaps[0])
        image, plan = imager.FIpipeDevice(ctx, pre["bin"], pre["vin"], pre["vis_re"], pre["vis_im"], case["size"],
                                          case["cell"], image=images[0], **opts)
        return {"image": image, "bin": pre["bin"], "vin": pre["vin"], "vis_re": pre["vis_re"],
                "vis_im": pre["vis_im"], "terms": plan["num_terms"], "slabs": plan["num_slabs"]}
    if call in ("single", "planned"):
        image, plan = imager.image_snapshot(ctx, snaps[0], case["size"], case["cell"], image=images[0],
                                            plan=state.get("plan"), **opts)
        return {"image": image, "terms": plan["num_terms"], "slabs": plan["num_slabs"]}
    if call == "batch":
        images, plans = imager.image_snapshot_batch(ctx, snaps, case["size"], case["cell"], images=images,
                                                    wait=False, **opts)
    else:
        images, plans = imager.image_snapshot_batch(ctx, snaps, state["sizes"], state["cells"], images=images, **opts)
    return {"images": images, "terms": [p["num_terms"] for p in plans], "slabs": [p["num_slabs"] for p in plans]}


def work(case):
    """Inputs read once and images written once; one complex-by-real multiply-add per footprint
    cell, term and unflagged sample, and 5 n log2 n operations per moment plane's transform."""
    nbytes = flops = 0.0
    for i in range(case["count"]):
        R, C = _num_rows(case, i), case["channels"]
        size, cell = _image(case, i)
        G = (3 * size + 1) // 2
        plan = _plan64(*_geometry(case, 0, i), size, cell, archive=case["call"] == "host")
        if case["call"] == "host":
            nbytes += 20.0 * R * C
        else:
            nbytes += (26.0 if case["weights"] else 18.0) * R * C + 24.0 * R + 8.0 * C
        if case["call"] == "pair":
            nbytes += 20.0 * R * C
        nbytes += 4.0 * size * size
        flops += 4.0 * 64 * plan["terms"] * R * C * (1.0 - case["flagged"])
        flops += 5.0 * plan["terms"] * plan["slabs"] * G * G * math.log2(G * G)
    return {"bytes": nbytes, "flops": flops}


# -------------------------------------------------------------------------- results in 64 bits

def _rotation64(uvw, freq):
    """Rows = the principal axes of the channel-folded baselines, largest variance first, with
    the reference's signs."""
    n = uvw.shape[0] * freq.numel()
    mean = uvw.sum(0) * freq.sum() / (C_LIGHT * n)
    scatter = (uvw.T @ uvw) * ((freq * freq).sum() / C_LIGHT ** 2) - n * torch.outer(mean, mean)
    v = torch.linalg.eigh(scatter.cpu())[1]
    r0, r1 = v[:, 2].clone(), v[:, 1].clone()
    if r0[0] < 0:
        r0 = -r0
    if r1[1] * ARRAY_CENTER_X < 0:
        r1 = -r1
    r2 = torch.linalg.cross(r0, r1)
    return torch.stack([r0, r1, r2 / torch.linalg.norm(r2)]).to(uvw.device)


def _fold64(snap, rot):
    """Rotated baselines (S, 3) in wavelengths and the weighted visibilities (S,), zero where both
    polarisations are flagged; sample = row + chan * rows."""
    b = ((snap["uvw"] @ rot.T)[None] * (snap["freq"] / C_LIGHT)[:, None, None]).reshape(-1, 3)
    num = torch.zeros(b.shape[0], dtype=torch.complex128, device=b.device)
    den = torch.zeros(b.shape[0], dtype=torch.float64, device=b.device)
    for pol in (0, 3):
        w = (snap[f"flag{pol}"] == 0).double()
        if snap[f"weight{pol}"] is not None:
            w = w * snap[f"weight{pol}"].double()
        num += w * torch.complex(snap[f"vis{pol}_re"].double(), snap[f"vis{pol}_im"].double())
        den += w
    return b, torch.where(den > 0, num / den.clamp(min=1e-30), torch.zeros_like(num))


def _bessel64(x, count, terms=48):
    """J_0 .. J_{count-1} by the power series, |x| <= 12."""
    h = x / 2.0
    lead, out = torch.ones_like(x), []
    for k in range(count):
        term, acc = lead, lead
        for m in range(1, terms):
            term = term * (-h * h) / (m * (m + k))
            acc = acc + term
        out.append(acc)
        lead = lead * h / (k + 1)
    return out


def _term_errors(alpha):
    """Largest error of the Chebyshev expansion of e^{i a s}, a <= alpha, per number of terms."""
    a = torch.linspace(0.0, alpha, 17, dtype=torch.float64)[:, None]
    s = torch.linspace(-1.0, 1.0, 513, dtype=torch.float64)[None, :]
    want, got, errs = torch.exp(1j * a * s), torch.zeros(17, 513, dtype=torch.complex128), []
    for k, j in enumerate(_bessel64(a, 32)):
        got = got + (2.0 if k else 1.0) * (1j ** k) * j * torch.cos(k * torch.arccos(s))
        errs.append(float((want - got).abs().max()))
    return errs


def _t3(rot, size, cell, idx):
    t = cell * (idx - size // 2).double()
    ra = 1.0 - (t[:, None] + rot[0, 2]) ** 2 - (t[None, :] + rot[1, 2]) ** 2
    sgn = 1.0 if float(rot[2, 2]) >= 0 else -1.0
    return torch.where(ra >= 0, -rot[2, 2] + sgn * torch.sqrt(ra.clamp(min=0.0)), torch.nan)


def _plan(rot, r3_min, r3_max, size, cell, archive):
    idx = torch.unique(torch.linspace(0, size - 1, min(size, 257)).round().long())
    t3 = float(torch.nan_to_num(_t3(rot, size, cell, idx)).abs().max())
    if archive:
        slabs, width, centre0 = 1, max(r3_max - r3_min, 2e-6), 0.5 * (r3_max + r3_min)
    else:
        width = max(r3_max - r3_min, 2e-6)
        slabs = max(1, math.ceil(2.0 * math.pi * t3 * max(0.5 * (r3_max - r3_min), 1e-6) / TARGET_ALPHA))
        width /= slabs
        centre0 = r3_min + 0.5 * width
    half = max(0.5 * width, 1e-6)
    alpha = 2.0 * math.pi * t3 * half
    errs = _term_errors(min(alpha, 12.0))
    options = range(1, 33) if archive else (8, 16, 24, 32)
    terms = next((k for k in options if errs[k - 1] <= TARGET_ERROR), 32)
    return {"slabs": slabs, "width": width, "half": half, "centre": centre0, "terms": terms, "alpha": alpha,
            "r3_min": r3_min}


def _plan64(uvw, freq, size, cell, archive=False):
    uvw, freq = torch.as_tensor(uvw), torch.as_tensor(freq)
    rot = _rotation64(uvw, freq)
    r3 = uvw @ rot[2]
    ends = torch.stack([r3 * float(freq.min()), r3 * float(freq.max())]) / C_LIGHT
    return _plan(rot.cpu(), float(ends.min()), float(ends.max()), size, cell, archive)


def _es64(x):
    return torch.where(x.abs() <= 1.0, torch.exp(BETA * (torch.sqrt((1.0 - x * x).clamp(min=0.0)) - 1.0)), 0.0)


def _grid64(p, vals, G):
    """(G, G, M): every sample's 8 x 8 ES footprint at p (S, 2) cells times its M values.  Samples
    near the centre, where a few cells take most of them, are summed as a dense product."""
    grid = torch.zeros(G * G, vals.shape[1], dtype=torch.float64, device=p.device)
    lo, hi, off = -(G // 2), (G - 1) // 2, G // 2
    B = min(96, G)
    b0 = -(B // 2)
    inner = ((p >= b0 + 4.0) & (p <= b0 + B - 5.0)).all(1)
    near, far = inner.nonzero().squeeze(1), (~inner).nonzero().squeeze(1)
    block = torch.zeros(B, B * vals.shape[1], dtype=torch.float64, device=p.device)
    cells = torch.arange(B, device=p.device, dtype=torch.float64) + b0
    step = max(256, (1 << 25) // (B * vals.shape[1]))
    for i in range(0, near.numel(), step):
        s = near[i:i + step]
        k1, k2 = (_es64((cells[None] - p[s, ax, None]) / 4.0) for ax in (0, 1))
        block += k1.T @ (k2[:, :, None] * vals[s][:, None, :]).reshape(s.numel(), -1)
    j = torch.arange(9, device=p.device, dtype=torch.float64)
    for i in range(0, far.numel(), 1 << 17):
        s = far[i:i + (1 << 17)]
        g = torch.ceil(p[s, :, None] - 4.0) + j
        k = _es64((g - p[s, :, None]) / 4.0) * ((g >= lo) & (g <= hi))
        g = (g.clamp(lo, hi) + off).long()
        w = (k[:, 0, :, None] * k[:, 1, None, :]).reshape(-1)
        at = (g[:, 0, :, None] * G + g[:, 1, None, :]).reshape(-1)
        who = torch.arange(s.numel(), device=p.device).repeat_interleave(81)
        nz = (w != 0).nonzero().squeeze(1)
        grid.index_add_(0, at[nz], w[nz, None] * vals[s][who[nz]])
    grid = grid.reshape(G, G, -1)
    grid[off + b0:off + b0 + B, off + b0:off + b0 + B] += block.reshape(B, B, -1)
    return grid


def _image64(b, vis, rot, plan, size, cell, signed, archive=False):
    """The image of rotated baselines and visibilities."""
    dev = b.device
    N, G, K = size, (3 * size + 1) // 2, plan["terms"]
    cell = float(np.float32(cell))
    half_n = N // 2
    n_samples = b.shape[0]
    keep = (vis != 0).nonzero().squeeze(1)
    b, vis = b[keep], vis[keep] / (rot[0, 0] * rot[1, 1] - rot[0, 1] * rot[1, 0]).abs()
    slab = ((b[:, 2] - plan["r3_min"]) / plan["width"]).floor().clamp(0, plan["slabs"] - 1)
    idx = torch.arange(N, device=dev)
    x = idx - half_n
    t3 = _t3(rot, N, cell, idx)
    valid = ~torch.isnan(t3)
    t3 = torch.nan_to_num(t3)
    J = _bessel64(2.0 * math.pi * t3 * plan["half"], K)
    g = torch.arange(G, device=dev)
    sign = 1.0 - 2.0 * ((g[:, None] + g[None, :] + 2 * (G // 2)) & 1).double()
    at = (G * G // 2 + G // 2 + x[:, None] * G + x[None, :]).reshape(-1)
    out = torch.zeros(N, N, dtype=torch.float64, device=dev)
    for ls in range(plan["slabs"]):
        centre = plan["centre"] + ls * plan["width"]
        m = (slab == ls).nonzero().squeeze(1)
        s = ((b[m, 2] - centre) / plan["half"]).clamp(-1.0, 1.0)
        v = torch.view_as_real(vis[m])
        vals = torch.cat([torch.cos(k * torch.arccos(s))[:, None] * v for k in range(K)], 1)
        grid = _grid64(b[m, :2] * (cell * G), vals, G)
        e = torch.exp(2j * math.pi * centre * t3)
        for k in range(K):
            f = torch.fft.ifft2(torch.view_as_complex(grid[..., 2 * k:2 * k + 2].contiguous()) * sign, norm="forward")
            out += ((2.0 if k else 1.0) * (1j ** k) * J[k] * e * f.reshape(-1)[at].reshape(N, N)).real
        del grid
    nodes, weights = (torch.from_numpy(a[14:].copy()).to(dev) for a in np.polynomial.legendre.leggauss(28))
    t = torch.arange(half_n + 1, device=dev).double()[:, None] / G
    conv = (_es64(nodes) * weights * torch.cos(math.pi * t * 8 * nodes)).sum(1) * 8 / CONV_NORM
    par = 1.0 - 2.0 * ((x[:, None] + x[None, :]) & 1).double()
    out = out * par / (conv[x.abs()][:, None] * conv[x.abs()][None, :] * CONV_NORM ** 2) / n_samples
    out = torch.where(valid, out, 0.0)
    return out if signed else _reproject64(out.abs(), valid, rot, N, cell, N // 2 if archive else N / 2.0)


def _reproject64(value, valid, rot, N, cell, mid):
    """|image| splatted bilinearly at each pixel's SIN re-projection (obliquity xi, eta)."""
    dev, c = value.device, N / 2.0
    y, x = (torch.arange(N, device=dev).double() - mid)[:, None], (torch.arange(N, device=dev).double() - mid)[None, :]
    p = [(-rot[0, i] * x + rot[1, i] * y) / rot[2, 2].abs() + (mid - c) for i in (0, 1)]
    px, py = -cell * (p[0] - 1.0), cell * (p[1] - 1.0)
    h2 = px * px + py * py
    z = h2 / (1.0 + torch.sqrt((1.0 - h2).clamp(min=0.0)))
    xi, eta = rot[2, 0] / rot[2, 2], rot[2, 1] / rot[2, 2]
    qx = torch.where(h2 <= 1.0, -(px + z * xi) / cell + 1.0, p[0]) + c - N // 2
    qy = torch.where(h2 <= 1.0, (py + z * eta) / cell + 1.0, p[1]) + c - N // 2
    ok = (valid & (qx.abs() < N // 2 - 1) & (qy.abs() < N // 2 - 1)).reshape(-1)
    qx, qy, value = qx.reshape(-1)[ok], qy.reshape(-1)[ok], value.reshape(-1)[ok]
    fx, fy = qx.floor(), qy.floor()
    out = torch.zeros(N * N, dtype=torch.float64, device=dev)
    for dx in (0, 1):
        for dy in (0, 1):
            w = (qx - fx if dx else 1.0 - qx + fx) * (qy - fy if dy else 1.0 - qy + fy)
            at = ((fy.long() + dy + N // 2) * N + fx.long() + dx + N // 2).clamp(0, N * N - 1)
            out.index_add_(0, at, w * value)
    return out.reshape(N, N)


def exact(case, seed):
    dev = torch.device("cuda", 0)
    size, cell = case["size"], case["cell"]
    archive = case["call"] == "host"
    if case["call"] in ("batch", "mixed"):
        return None
    plan = _plan64(*_geometry(case, seed, 0), size, cell, archive=archive)
    if 64.0 * _num_rows(case) * case["channels"] * 2 * plan["terms"] > EXACT_LIMIT:
        return None
    if archive:
        b, rot, re, im = (t.double() for t in _host_samples(case, seed, dev))
        plan = _plan(rot.cpu(), float(b[:, 2].min()), float(b[:, 2].max()), size, cell, True)
        return {"image": _image64(b, torch.complex(re, im), rot, plan, size, cell, case["signed"], True), "terms": None}
    snap = _snapshot(case, seed, 0, dev)
    rot = _rotation64(snap["uvw"], snap["freq"])
    b, vis = _fold64(snap, rot)
    out = {"image": _image64(b, vis, rot, plan, size, cell, case["signed"]), "terms": None, "slabs": None}
    if case["call"] == "pair":
        out.update(bin=b, vin=rot, vis_re=vis.real, vis_im=vis.imag)
    return out

"""Performance cases: the scoring work a program gives this framework, through
its public entry points.

A case is one call of a kind of program:

    pipeline  one pair in device memory through ``Ssimulacra2Pipeline.Compute``:
              an encoder's rate control or a viewer that scores one frame and
              waits for it
    batch     device-resident pairs through ``Ssimulacra2Batch``: a sweep over
              encoded frames, every pair of one size or of several
    server    a burst of requests of mixed sizes through ``Ssimulacra2Server``
    pool      host images through ``Ssimulacra2Pool``, uploads included: a
              command that scores decoded files

``input`` is the pixel format: ``srgb8`` (8-bit sRGB RGB planes), ``yuv420``
(8-bit limited-range BT.709 4:2:0, decoded video) or ``pq420`` (10-bit
limited-range BT.2020 PQ 4:2:0 in 16-bit words, HDR video). ``planes`` is the
stored plane format (``f32`` the default, ``f16`` the half-plane build, ``u16``
the mixed form) and ``map`` the arithmetic form (0 default, 1 reference, 2
difference).

    listed()              the cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   the inputs and the engine a program holds before the call
    run(state)            one call: the 108 norms of every pair, FP64
    work(case)            bytes and operations one call cannot do without
    exact(case, seed)     the norms computed in 64 bits by plain torch
"""
from __future__ import annotations

import math

import numpy as np
import torch

from vqm_amd import (ColorFamily, ColorPrimaries, DeviceImage, Image, ImageFormat, MatrixCoefficients,
                     PixelRange, PixelType, Size, Ssimulacra2Batch, Ssimulacra2Config, Ssimulacra2Pipeline,
                     Ssimulacra2Pool, Ssimulacra2Server, TransferCharacteristics)

PLANES = {"f32": 0, "f16": 1, "u16": 3}
LADDER = "640x360,1280x720,1920x1080,2560x1440,3840x2160"
POOL_WORKERS = 3
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def case_(name, kind, size, pairs=1, input="srgb8", planes="f32", map=0):
    return {"name": name, "kind": kind, "size": size, "pairs": pairs, "input": input, "planes": planes, "map": map}


def listed():
    return [
        # A thumbnail pair: launches and latency are all of it.
        case_("pair_96x64", "pipeline", "96x64"),
        # The single 512x512 image pair of codec comparisons.
        case_("pair_512", "pipeline", "512x512"),
        # One video frame pair, waited for: per-frame quality control.
        case_("pair_1080p", "pipeline", "1920x1080"),
        # One UHD frame pair.
        case_("pair_4k", "pipeline", "3840x2160"),
        # A decoded 8-bit video frame pair (general per-pixel decode).
        case_("pair_yuv420_1080p", "pipeline", "1920x1080", input="yuv420"),
        # A decoded HDR10 frame pair.
        case_("pair_pq420_4k", "pipeline", "3840x2160", input="pq420"),
        # Host images: uploads overlap the kernels of three pipelines.
        case_("pool_host_1080p_6", "pool", "1920x1080", pairs=6),
        # A small batch of an odd size (rows that are not 4-byte aligned).
        case_("batch_853x479_8", "batch", "853x479", pairs=8),
        # The headline: 300 resident 1080p pairs a call.
        case_("batch_1080p_300", "batch", "1920x1080", pairs=300),
        # The mixed form: 16-bit fixed-point planes, difference arithmetic.
        case_("batch_1080p_u16_100", "batch", "1920x1080", pairs=100, planes="u16"),
        # A batch of uneven sizes, 640x360 to 4K.
        case_("batch_ladder_60", "batch", LADDER, pairs=60),
        # A burst of 64 requests of the same sizes against the server.
        case_("serve_ladder_64", "server", LADDER, pairs=64),
    ]


def log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["pipeline", "pipeline", "pipeline", "batch", "batch", "pool", "server"])
    input, planes, map_ = "srgb8", "f32", 0
    if kind in ("pipeline", "pool"):
        input = rng.choice(["srgb8", "srgb8", "yuv420", "pq420"])
    if kind != "pool":
        planes = rng.choice(["f32", "f32", "f32", "u16", "f16"])
        map_ = 2 if planes == "f32" and rng.random() < 0.25 else 0
    if kind == "server" or (kind == "batch" and rng.random() < 0.4):
        sizes = ["%dx%d" % (log_uniform(rng, 256, 3840), log_uniform(rng, 256, 2160))
                 for _ in range(rng.randint(2, 5))]
        return {"kind": kind, "size": ",".join(sizes), "pairs": rng.randint(4, 48), "input": input,
                "planes": planes, "map": map_}
    w, h = log_uniform(rng, 64, 3840), log_uniform(rng, 64, 2160)
    if input != "srgb8":  # 4:2:0 frames have even sides
        w, h = w + w % 2, h + h % 2
    pairs = 1
    if kind == "batch":
        pairs = log_uniform(rng, 1, min(300, 100 * 1920 * 1080 / (w * h)))
    elif kind == "pool":
        pairs = rng.randint(3, 6)
    return {"kind": kind, "size": "%dx%d" % (w, h), "pairs": pairs, "input": input, "planes": planes, "map": map_}


def sizes_of(case):
    """(width, height) of every pair: the case's sizes in turn."""
    sizes = [tuple(int(v) for v in s.split("x")) for s in case["size"].split(",")]
    return [sizes[i % len(sizes)] for i in range(case["pairs"])]


# ---- inputs -------------------------------------------------------------------

def format_of(input):
    if input == "srgb8":
        return ImageFormat.srgb8()
    if input == "yuv420":
        return ImageFormat(type=PixelType.Byte, family=ColorFamily.Yuv, range=PixelRange.Limited,
                           matrix=MatrixCoefficients.Bt709, transfer=TransferCharacteristics.Bt709,
                           primaries=ColorPrimaries.Bt709, subsample_w=1, subsample_h=1)
    return ImageFormat(type=PixelType.Word, family=ColorFamily.Yuv, range=PixelRange.Limited,
                       matrix=MatrixCoefficients.Bt2020Ncl, transfer=TransferCharacteristics.St2084,
                       primaries=ColorPrimaries.Bt2020, subsample_w=1, subsample_h=1, depth=10)


def plane_sizes(input, w, h):
    return [(w, h)] * 3 if input == "srgb8" else [(w, h), (w // 2, h // 2), (w // 2, h // 2)]


def field(gen, w, h, extent):
    """A smooth picture in [0, 1]: a ramp and four sinusoids of 8 to 512 pixels."""
    p = torch.rand(16, generator=gen, dtype=torch.float64).tolist()
    x = torch.arange(w, device=DEVICE, dtype=torch.float32)[None, :] * (extent / w)
    y = torch.arange(h, device=DEVICE, dtype=torch.float32)[:, None] * (extent / h)
    v = 0.5 + 0.2 * (p[0] - 0.5) * x / extent + 0.2 * (p[1] - 0.5) * y / extent
    for k in range(4):
        period = 8.0 * 64.0 ** p[2 + 3 * k]
        angle = 2.0 * math.pi * p[3 + 3 * k]
        f = 2.0 * math.pi / period
        v = v + 0.11 * torch.sin(f * math.cos(angle) * x + f * math.sin(angle) * y + 6.28 * p[4 + 3 * k])
    return v


# What each format's planes hold: the range of the codes of a picture, the
# largest code, and the noise sigma of one distortion step.
CODES = {"srgb8": ([(0, 255)] * 3, 255, 1.0),
         "yuv420": ([(16, 235), (80, 176), (80, 176)], 255, 1.0),
         "pq420": ([(120, 720), (440, 584), (440, 584)], 1023, 3.0)}
STRENGTHS = ((4, 1.0), (12, 3.0), (24, 8.0))  # quantisation step, noise sigma


def pair_planes(case, index, w, h, seed):
    """Integer code planes of the original and of its distorted copy (each
    8x8 block quantised around its corner sample, and noise), as a codec
    leaves them."""
    input = case["input"]
    ranges, top, unit = CODES[input]
    gen = torch.Generator().manual_seed(seed * 1000003 + index * 7919 + 17)
    noise = torch.Generator(device=DEVICE).manual_seed(seed * 1000003 + index * 7919 + 29)
    step, sigma = STRENGTHS[index % len(STRENGTHS)]
    a, b = [], []
    for (pw, ph), (low, high) in zip(plane_sizes(input, w, h), ranges):
        v = low + (high - low) * field(gen, pw, ph, float(w))
        v = v + unit * torch.randn((ph, pw), generator=noise, device=DEVICE)
        o = v.round().clamp(0, top)
        corner = o[(torch.arange(ph, device=DEVICE) // 8 * 8)][:, (torch.arange(pw, device=DEVICE) // 8 * 8)]
        q = unit * step
        d = corner + ((o - corner) / q).round() * q
        d = d + unit * sigma * torch.randn((ph, pw), generator=noise, device=DEVICE)
        a.append(o)
        b.append(d.round().clamp(0, top))
    return a, b


def pack(input, planes):
    """Packed planes, each on a 4-byte boundary, as a uint8 tensor."""
    parts = []
    for p in planes:
        flat = p.reshape(-1)
        raw = flat.to(torch.uint8) if input != "pq420" else flat.to(torch.int16).view(torch.uint8)
        pad = -raw.numel() % 4
        parts.append(raw)
        if pad:
            parts.append(torch.zeros(pad, dtype=torch.uint8, device=raw.device))
    return torch.cat(parts)


def prepare(case, seed):
    sizes = sizes_of(case)
    images = []
    for i, (w, h) in enumerate(sizes):
        a, b = pair_planes(case, i, w, h, seed)
        images.append((pack(case["input"], a), pack(case["input"], b)))
    planes, map_ = PLANES[case["planes"]], case["map"]
    fmt = format_of(case["input"])
    state = {"kind": case["kind"], "images": images}
    if case["kind"] in ("pipeline", "pool"):
        size = Size(*sizes[0])
        streaming = case["kind"] == "pool"
        config = Ssimulacra2Config(size=size, gpu_resident_images=0, streaming_inputs=streaming,
                                   plane_format=planes, map_form=map_)
        if streaming:
            state["engine"] = Ssimulacra2Pool(config, POOL_WORKERS)
            state["pairs"] = [tuple(Image(size, fmt, x.cpu().numpy()) for x in p) for p in images]
            state["images"] = None
        else:
            state["engine"] = Ssimulacra2Pipeline(config)
            state["pairs"] = [tuple(DeviceImage(x.data_ptr(), size, fmt, x.numel()) for x in p) for p in images]
        return state
    if case["kind"] == "batch":
        state["engine"] = Ssimulacra2Batch(len(sizes), plane_format=planes, map_form=map_)
        state["pairs"] = [(a.data_ptr(), b.data_ptr(), w, h) for (a, b), (w, h) in zip(images, sizes)]
    else:
        state["engine"] = Ssimulacra2Server(plane_format=planes, map_form=map_)
        state["pairs"] = [(a.data_ptr(), b.data_ptr(), w, h, False, 0) for (a, b), (w, h) in zip(images, sizes)]
    return state


def run(state):
    engine, pairs = state["engine"], state["pairs"]
    if state["kind"] == "pipeline":
        return engine.Compute(*pairs[0]).norms()
    if state["kind"] == "pool":
        return np.stack([r.norms() for r in engine.ComputeMany(pairs)])
    if state["kind"] == "batch":
        return engine.Finish(engine.Submit(pairs), raw=True)[1]
    return np.stack([r.norms for r in engine.Replay(pairs)])


# ---- the work of a call ---------------------------------------------------------

# Channels (bit 0 X, 1 Y, 2 B) that carry score weight at each level, by the
# number of levels: the metric scores no others, and their norms are zero.
ACTIVE = {1: (6,), 2: (6, 3), 3: (6, 7, 5), 4: (6, 5, 7, 3), 5: (4, 3, 3, 3, 3), 6: (2, 3, 3, 7, 7, 0)}


def levels_of(w, h):
    out = []
    while len(out) < 6:
        out.append((w, h))
        if w < 8 or h < 8:
            break
        w, h = (w + 1) // 2, (h + 1) // 2
    return out


def work(case):
    nbytes = flops = 0
    sample = 2 if case["input"] == "pq420" else 1
    for w, h in sizes_of(case):
        nbytes += 2 * sample * sum(pw * ph for pw, ph in plane_sizes(case["input"], w, h)) + 108 * 8
        levels = levels_of(w, h)
        for (lw, lh), mask in zip(levels, ACTIVE[len(levels)]):
            # Both images: box, two or three opsin mixes and cube roots a pixel.
            flops += 2 * 60 * lw * lh
            # A scored plane: products, five quantities through two 13-tap
            # passes, the two maps and their six sums.
            flops += bin(mask).count("1") * (3 + 5 * 2 * 25 + 40) * lw * lh
    return {"bytes": nbytes, "flops": flops}


# ---- 64 bits ---------------------------------------------------------------------

def srgb_eotf(v):
    return torch.where(v <= 0.04045, v / 12.92, ((v + 0.055) / 1.055).clamp(min=0) ** 2.4)


def pq_eotf(v):
    """SMPTE ST 2084, over a 100 cd/m2 white."""
    m1, m2 = 2610.0 / 16384.0, 2523.0 / 4096.0 * 128.0
    c1, c2, c3 = 3424.0 / 4096.0, 2413.0 / 4096.0 * 32.0, 2392.0 / 4096.0 * 32.0
    p = v.clamp(min=0) ** (1.0 / m2)
    return 100.0 * ((p - c1).clamp(min=0) / (c2 - c3 * p)) ** (1.0 / m1)


def upsample_left(plane, w, h):
    """4:2:0 chroma, left-sited, bilinear with mirrored edges."""
    def axis(n, out, shift):
        pos = (torch.arange(out, device=DEVICE, dtype=torch.float64) + 0.5) / 2.0 + shift
        first = torch.floor(pos - 0.5)
        t = pos - (first + 0.5)
        # A tap's centre is mirrored at the plane's edges: sample -1 is sample 0,
        # and sample n is sample n - 1.
        i0, i1 = first.long().clamp(0, n - 1), (first.long() + 1).clamp(0, n - 1)
        return i0, i1, t
    x0, x1, tx = axis(plane.shape[1], w, 0.25)
    y0, y1, ty = axis(plane.shape[0], h, 0.0)
    rows = plane[:, x0] * (1 - tx) + plane[:, x1] * tx
    return rows[y0] * (1 - ty)[:, None] + rows[y1] * ty[:, None]


def ncl(kr, kb, y, u, v):
    """Non-constant-luminance Y'CbCr to R'G'B'."""
    r = y + 2.0 * (1.0 - kr) * v
    b = y + 2.0 * (1.0 - kb) * u
    return [r, (y - kr * r - kb * b) / (1.0 - kr - kb), b]


def rgb_to_xyz(primaries):
    xyz = torch.tensor([[x / y, 1.0, (1.0 - x - y) / y] for x, y in primaries], dtype=torch.float64).T
    white = torch.tensor([0.3127 / 0.3290, 1.0, (1.0 - 0.3127 - 0.3290) / 0.3290], dtype=torch.float64)
    return xyz * torch.linalg.solve(xyz, white)[None, :]


def linear(input, planes, w, h):
    """Linear BT.709 RGB of code planes."""
    planes = [p.double() for p in planes]
    if input == "srgb8":
        return [srgb_eotf(p / 255.0) for p in planes]
    depth = 8 if input == "yuv420" else 10
    unit = float(1 << (depth - 8))
    y = (planes[0] - 16.0 * unit) / (219.0 * unit)
    u, v = [upsample_left((p - 128.0 * unit) / (224.0 * unit), w, h) for p in planes[1:]]
    if input == "yuv420":
        return [c.clamp(min=0) ** 2.4 for c in ncl(0.2126, 0.0722, y, u, v)]
    rgb = [pq_eotf(c) for c in ncl(0.2627, 0.0593, y, u, v)]
    m = torch.linalg.solve(rgb_to_xyz([(0.640, 0.330), (0.300, 0.600), (0.150, 0.060)]),
                           rgb_to_xyz([(0.708, 0.292), (0.170, 0.797), (0.131, 0.046)])).tolist()
    return [row[0] * rgb[0] + row[1] * rgb[1] + row[2] * rgb[2] for row in m]


def xyb(rgb):
    """The metric's opsin transform, offset to positive values."""
    bias = 0.0037930732552754493
    rows = ((0.30, 0.622, 0.078), (0.23, 0.692, 0.078),
            (0.24342268924547819, 0.20476744424496821, 1.0 - 0.24342268924547819 - 0.20476744424496821))
    c = [(r[0] * rgb[0] + r[1] * rgb[1] + r[2] * rgb[2] + bias).clamp(min=0) ** (1.0 / 3.0) - bias ** (1.0 / 3.0)
         for r in rows]
    y = 0.5 * (c[0] + c[1])
    return [0.5 * (c[0] - c[1]) * 14.0 + 0.42, y + 0.01, c[2] - y + 0.55]


def half(p):
    """The 2x2 box mean, the last row and column repeated on odd sides."""
    h, w = p.shape
    if w % 2:
        p = torch.cat([p, p[:, -1:]], 1)
    if h % 2:
        p = torch.cat([p, p[-1:]], 0)
    return 0.25 * (p[0::2, 0::2] + p[0::2, 1::2] + p[1::2, 0::2] + p[1::2, 1::2])


def blur(x, taps):
    h, w = x.shape[-2:]
    x = torch.nn.functional.pad(x, (6, 6))
    x = sum(t * x[..., k:k + w] for k, t in enumerate(taps))
    x = torch.nn.functional.pad(x, (0, 0, 6, 6))
    return sum(t * x[..., k:k + h, :] for k, t in enumerate(taps))


def pair_norms(input, a, b, w, h):
    taps = [math.exp(-0.5 * ((k - 6) / 1.5) ** 2) for k in range(13)]
    taps = [t / sum(taps) for t in taps]
    norms = torch.zeros(108, dtype=torch.float64)
    la, lb = linear(input, a, w, h), linear(input, b, w, h)
    levels = levels_of(w, h)
    for level, mask in enumerate(ACTIVE[len(levels)]):
        if level:
            la, lb = [half(p) for p in la], [half(p) for p in lb]
        if not mask:
            continue
        xa, xb = xyb(la), xyb(lb)
        for c in range(3):
            if not mask >> c & 1:
                continue
            p, q = xa[c], xb[c]
            mu1, mu2, s11, s22, s12 = blur(torch.stack([p, q, p * p, q * q, p * q]), taps)
            num_m = 1.0 - (mu1 - mu2) ** 2
            num_s = 2.0 * (s12 - mu1 * mu2) + 0.0009
            den = (s11 - mu1 * mu1) + (s22 - mu2 * mu2) + 0.0009
            d = (1.0 - num_m * num_s / den).clamp(min=0)
            e = (1.0 + (q - mu2).abs()) / (1.0 + (p - mu1).abs()) - 1.0
            ring, soft = e.clamp(min=0), (-e).clamp(min=0)
            v = []
            for m in (d, ring, soft):
                v += [m.mean(), (m ** 4).mean() ** 0.25]
            v = torch.stack(v).cpu()
            norms[18 * level + 2 * c:18 * level + 2 * c + 2] = v[:2]
            norms[18 * level + 6 + 4 * c:18 * level + 6 + 4 * c + 4] = v[2:]
    return norms


def exact(case, seed):
    if case["planes"] == "f16":
        return None  # the half-plane build's norms are those of rounded planes
    out = []
    for i, (w, h) in enumerate(sizes_of(case)):
        a, b = pair_planes(case, i, w, h, seed)
        out.append(pair_norms(case["input"], a, b, w, h))
    return out[0].numpy() if case["kind"] == "pipeline" else torch.stack(out).numpy()

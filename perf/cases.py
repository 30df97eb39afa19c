"""Performance cases of the denoising core: what is timed, on which inputs, through which entry points.

A case is a dict of plain values; ``prepare`` builds what a program holds before the call, ``run``
makes one pass through the public entry points and returns its outputs, ``work`` states the bytes
and operations the pass cannot do without, ``exact`` the outputs in 64 bits where they are numbers
rather than sample codes.

The kinds:

* ``nlmeans`` and ``nl4d``: one frame of a running stream through the engine (``push`` and
  ``emit_into`` of device planes), the window already full.  Outputs are the planes' bytes.
* ``host``: the same over host bytes (``HostDenoiser``), one frame kept in flight.
* ``noise``: the noise measurements of one frame (spatial totals and temporal block records).
* ``grain``: the film-grain measurements of one completed frame (vector save, measure, reduce,
  projection, persistence).
* ``grain_fit``: the AR(3) fit of a segment's pooled records.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "av-denoise_amd"))

import avd  # noqa: E402
from avd._lib import check  # noqa: E402

CHROMA = {"gray": 0, "420": 1, "422": 2, "444": 3}
CLIP_FRAMES = 12


def listed():
    return [
        # A web-sized clip, luma only: the plain spatial filter with a wide window (latency, few waves).
        {"name": "nlm_spatial_360p", "kind": "nlmeans", "width": 640, "height": 360, "chroma": "gray", "depth": 8,
         "hq": False, "radius": 0, "patch": 2, "search": 7, "motion": False},
        # Full HD 10-bit with temporal neighbours: the plain filter's ordinary work.
        {"name": "nlm_temporal_1080p", "kind": "nlmeans", "width": 1920, "height": 1080, "chroma": "420", "depth": 10,
         "hq": False, "radius": 2, "patch": 3, "search": 4, "motion": False},
        # The "base" preset (HQ, block confidence, no warp) on 8-bit full HD.
        {"name": "nlm_hq_base_1080p", "kind": "nlmeans", "width": 1920, "height": 1080, "chroma": "420", "depth": 8,
         "hq": True, "radius": 2, "patch": 4, "search": 2, "motion": False},
        # HQ with motion compensation over a long window, an odd-sized 4:2:2 crop.
        {"name": "nlm_hq_motion_odd", "kind": "nlmeans", "width": 1277, "height": 717, "chroma": "422", "depth": 10,
         "hq": True, "radius": 4, "patch": 4, "search": 4, "motion": True},
        # NL4D on the dense grid in the matrix-core form at 4K: the largest frames, the quality setting.
        {"name": "nl4d_dense_4k", "kind": "nl4d", "width": 3840, "height": 2160, "chroma": "420", "depth": 10,
         "radius": 3, "spatial": 12, "step": 3, "group": 16, "mixed": True, "pooled": False},
        # NL4D's defaults (stride 4, groups of 8, pooled threshold, FP32 form) on 8-bit full HD.
        {"name": "nl4d_base_1080p", "kind": "nl4d", "width": 1920, "height": 1080, "chroma": "420", "depth": 8,
         "radius": 2, "spatial": 9, "step": 4, "group": 8, "mixed": False, "pooled": True},
        # A small odd-sized 4:4:4 clip through NL4D: many launches, little work in each.
        {"name": "nl4d_small_odd", "kind": "nl4d", "width": 427, "height": 241, "chroma": "444", "depth": 10,
         "radius": 1, "spatial": 9, "step": 4, "group": 8, "mixed": False, "pooled": False},
        # A file converter's loop: host bytes in, host bytes out, the "veryfast" preset at 720p.
        {"name": "host_nlm_720p", "kind": "host", "engine": "nlmeans", "width": 1280, "height": 720, "chroma": "420",
         "depth": 8, "hq": False, "radius": 0, "patch": 4, "search": 2, "motion": False},
        # Noise measurement of a 4K luma frame against the previous one, along the motion field.
        {"name": "noise_luma_4k", "kind": "noise", "width": 3840, "height": 2160, "channels": 1, "motion": True},
        # Noise measurement of a small odd chroma pair at the zero vector.
        {"name": "noise_chroma_odd", "kind": "noise", "width": 477, "height": 269, "channels": 2, "motion": False},
        # Film-grain measurement of a completed full HD luma frame.
        {"name": "grain_1080p", "kind": "grain", "width": 1920, "height": 1080, "channels": 1},
        # The AR fit of a segment: one record per strength group.
        {"name": "grain_fit_16", "kind": "grain_fit", "records": 16},
    ]


def _size(rng, lo, hi, least=64):
    """A frame size between lo and hi columns, uniform over the logarithm, odd ones among them."""
    w = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    h = max(least, int(w * rng.choice([9 / 16, 3 / 4, 9 / 21]) + rng.randrange(-3, 4)))
    return w, h


def draw(rng):
    kind = rng.choice(["nlmeans", "nlmeans", "nlmeans", "nl4d", "nl4d", "nl4d", "host", "noise", "noise", "grain",
                       "grain_fit"])
    if kind == "grain_fit":
        return {"kind": kind, "records": rng.randrange(1, 65)}
    chroma, depth = rng.choice(["gray", "420", "422", "444"]), rng.choice([8, 10, 10, 12])
    if kind == "noise":
        w, h = _size(rng, 200, 3840)
        return {"kind": kind, "width": w, "height": h, "channels": rng.choice([1, 2]),
                "motion": rng.choice([True, False])}
    if kind == "grain":
        w, h = _size(rng, 320, 3840)
        return {"kind": kind, "width": w, "height": h, "channels": rng.choice([1, 2])}
    if kind == "nl4d":
        mixed = rng.choice([True, False])
        w, h = _size(rng, 200, 2560)
        return {"kind": kind, "width": w, "height": h, "chroma": chroma, "depth": depth, "radius": rng.choice([1, 2, 3]),
                "spatial": rng.choice([9, 12]), "step": rng.choice([3, 4, 4]), "group": rng.choice([8, 16]),
                "mixed": mixed, "pooled": False if mixed else rng.choice([True, False])}
    hq = rng.choice([True, False])
    radius = rng.choice([1, 2, 4]) if hq else rng.choice([0, 0, 1, 2])
    if kind == "host":
        radius = min(radius, 2)
    w, h = _size(rng, 200, 1920 if radius <= 2 else 1280)
    case = {"kind": kind, "width": w, "height": h, "chroma": chroma, "depth": depth, "hq": hq, "radius": radius,
            "patch": rng.choice([1, 2, 3, 4]), "search": rng.choice([2, 3, 4, 7 if radius == 0 else 4]),
            "motion": rng.choice([True, False]) if hq else False}
    if kind == "host":
        case["engine"] = "nlmeans"
    return case


# ---- inputs -----------------------------------------------------------------------------------


def _sigma(case):
    """The clip's noise in codes of its depth: light sensor noise, the same strength at any depth."""
    scale = (1 << case["depth"]) / 1024.0
    return 14.0 * scale, 8.0 * scale


def _scene(rng, frames, width, height, shift, scale_x, scale_y):
    """`frames` pictures of a moving scene in 0..1: slow shading, oriented texture and hard edges."""
    dev = "cuda"
    periods = rng.uniform(8.0, 128.0, 6)
    theta = rng.uniform(0.0, math.pi, 6)
    phase = rng.uniform(0.0, 2.0 * math.pi, 6)
    amp = rng.uniform(0.3, 1.0, 6)
    edge = rng.uniform(0.0, 2.0 * math.pi, 4)
    ys = torch.arange(height, device=dev, dtype=torch.float32).unsqueeze(1) * scale_y
    xs = torch.arange(width, device=dev, dtype=torch.float32).unsqueeze(0) * scale_x
    out = []
    for t in range(frames):
        x, y = xs + float(shift[t, 0]), ys + float(shift[t, 1])
        acc = torch.zeros(height, width, device=dev)
        for p, th, ph, a in zip(periods, theta, phase, amp):
            acc += a * torch.sin((2.0 * math.pi / p) * (x * math.cos(th) + y * math.sin(th)) + ph)
        # Texture fades out over large flat areas, and two sets of edges cut the picture.
        mask = torch.sigmoid(4.0 * torch.sin(x / 211.0 + edge[0]) * torch.sin(y / 173.0 + edge[1]))
        bars = torch.sign(torch.sin(x / 37.0 + edge[2]) + torch.sin(y / 53.0 + edge[3]))
        out.append(0.5 + 0.09 * acc * mask + 0.06 * bars + 0.12 * torch.sin(x / 401.0 + y / 307.0))
    return out


def _planes(case):
    w, h = case["width"], case["height"]
    c = avd.chroma_dims(CHROMA[case["chroma"]], w, h)
    return [(w, h)] + ([c, c] if c else [])


def _clip(case, seed, frames):
    """Frames of integer code planes on the GPU, from the seed alone."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    depth = case["depth"]
    top, lo, hi = (1 << depth) - 1, 16 << (depth - 8), 235 << (depth - 8)
    shift = np.cumsum(rng.integers(-4, 5, size=(frames, 2)), axis=0) + 0.25 * np.arange(frames)[:, None]
    dims, noise = _planes(case), _sigma(case)
    planes = []
    for k, (w, h) in enumerate(dims):
        sx, sy = case["width"] / w, case["height"] / h
        pics = _scene(rng, frames, w, h, shift, sx, sy)
        sigma = noise[0] if k == 0 else noise[1]
        planes.append([torch.clamp(torch.round(lo + p.clamp(0, 1) * (hi - lo) +
                                               torch.randn(h, w, device="cuda", generator=gen) * sigma), 0, top)
                       .to(torch.int32) for p in pics])
    return [list(f) for f in zip(*planes)]


def _pack(codes, depth):
    """A code plane as the engine's device plane: samples in order, padded to a whole 32-bit word."""
    flat = codes.reshape(-1).to(torch.uint8 if depth == 8 else torch.int16).view(torch.uint8)
    out = torch.zeros((flat.numel() + 3) // 4 * 4, dtype=torch.uint8, device=flat.device)
    out[:flat.numel()] = flat
    return out


def _engine_parts(case):
    fmt = avd.SampleFormat.u8() if case["depth"] == 8 else avd.SampleFormat.u16(case["depth"])
    geom = avd.Geometry(case["width"], case["height"], CHROMA[case["chroma"]], fmt, fmt, 0)
    top = float((1 << case["depth"]) - 1)
    noise = [s / top for s in _sigma(case)]

    def options(k):
        if case["kind"] == "nl4d":
            return avd.nl4d_options(temporal_radius=case["radius"], spatial_radius=case["spatial"], step=case["step"],
                                    group_size=case["group"], transform_form=1 if case["mixed"] else 0,
                                    pooled_threshold=1 if case["pooled"] else 0, noise_map=0, field_lambda=0.0,
                                    sigma=noise[k], motion={"estimation": 1},
                                    **({} if case["pooled"] else {"lambda_ht": 2.7}))
        o = dict(hq=1 if case["hq"] else 0, temporal=1 if case["radius"] else 0, temporal_radius=case["radius"],
                 patch_radius=case["patch"], search_radius=case["search"],
                 motion_compensation=1 if case["motion"] else 0, motion={"estimation": 1})
        if case["hq"]:
            o["sigma"] = noise[k]
        else:
            o["strength"] = 1.2
        return avd.nlmeans_options(**o)

    chroma = None if case["chroma"] == "gray" else options(1)
    return geom, options(0), chroma


def _emitted(eng, state):
    for _ in range(eng.push(state["frames"][state["at"] % len(state["frames"])])):
        eng.emit_into(state["outs"])
    state["at"] += 1


def _prepare_stream(case, seed):
    geom, luma, chroma = _engine_parts(case)
    eng = avd.build_engine(case["kind"], geom, luma=luma, chroma=chroma)
    frames = [[_pack(p, case["depth"]) for p in f] for f in _clip(case, seed, CLIP_FRAMES)]
    outs = [torch.zeros(avd.plane_bytes(geom.output, w, h), dtype=torch.uint8, device="cuda") for w, h in _planes(case)]
    state = {"kind": case["kind"], "engine": eng, "frames": frames, "outs": outs, "at": 0}
    for _ in range(2 * case["radius"] + 1):  # the window fills; every later push readies one frame
        _emitted(eng, state)
    return state


def _prepare_host(case, seed):
    geom, luma, chroma = _engine_parts(case)
    den = avd.HostDenoiser(case["engine"], geom, luma=luma, chroma=chroma)
    kind = np.uint8 if case["depth"] == 8 else np.uint16
    frames = [[p.cpu().numpy().astype(kind).reshape(-1).view(np.uint8) for p in f]
              for f in _clip(case, seed, CLIP_FRAMES)]
    state = {"kind": "host", "engine": den, "frames": frames, "at": 0}
    while den.pending() < 1:
        den.push(frames[state["at"] % CLIP_FRAMES])
        state["at"] += 1
    return state


# ---- measurement sites -------------------------------------------------------------------------


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _noise_inputs(case, seed):
    """A two-frame ring of normalised samples, slot 1 the new frame, and a motion field on the
    8-pixel grid that mostly follows the scene's pan."""
    W, H, C = case["width"], case["height"], case["channels"]
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    pan = rng.integers(-4, 5, size=2)
    shift = np.stack([np.zeros(2), pan]).astype(np.float64)
    ring = torch.empty(2, H, W, C, device="cuda")
    for c in range(C):
        for f, pic in enumerate(_scene(rng, 2, W, H, shift, 1.0, 1.0)):
            ring[f, :, :, c] = (pic + torch.randn(H, W, device="cuda", generator=gen) * 0.01).clamp(0, 1)
    bx, by = -(-W // 8), -(-H // 8)
    field = None
    if case["motion"]:
        # Most blocks hold the pan, a tenth a vector of their own and a fifth none.
        pick = torch.rand(by, bx, 1, device="cuda", generator=gen)
        own = torch.randint(-9, 10, (by, bx, 2), device="cuda", generator=gen, dtype=torch.int32)
        base = torch.tensor([int(pan[0]), int(pan[1])], device="cuda", dtype=torch.int32).expand(by, bx, 2)
        field = torch.where(pick < 0.1, own, torch.where(pick < 0.3, torch.zeros_like(own), base)).contiguous()
    return ring.contiguous(), field, bx, by


def _record_parts(stats, C):
    """The block records' lanes by meaning, as views: sums, textures and the moved flag; the
    quarters' sums; their flatness (3e38 where unmeasured); their extremes."""
    v = stats.view(-1, 3 * C + 26)
    q = v[:, 2 * C + 3:2 * C + 27].unflatten(1, (4, 6))
    return {"head": v[:, :2 * C + 3], "quarter_sums": q[:, :, :3], "flatness": q[:, :, 3], "extremes": q[:, :, 4:],
            "tail": v[:, 2 * C + 27:]}


def _prepare_noise(case, seed):
    W, H, C = case["width"], case["height"], case["channels"]
    lib = avd.load()
    ring, field, bx, by = _noise_inputs(case, seed)
    stats = torch.zeros(lib.avd_noise_temporal_stats_len(W, H, C), device="cuda")
    state = {"kind": "noise", "case": case, "lib": lib, "ring": ring, "field": field, "grid": (bx, by),
             "partials": torch.empty(lib.avd_noise_partials_len(W, H), device="cuda"),
             "totals": torch.zeros(2, device="cuda"), "stats": stats}
    state["out"] = {"totals": state["totals"], **_record_parts(stats, C)}
    return state


def _run_noise(s):
    c, lib, st = s["case"], s["lib"], _stream()
    bx, by = s["grid"]
    check(lib.avd_site_noise_spatial(_ptr(s["ring"]), c["width"], c["height"], c["channels"], 1, _ptr(s["partials"]),
                                     _ptr(s["totals"]), 0, st))
    check(lib.avd_site_noise_temporal_stats(_ptr(s["ring"]), c["width"], c["height"], c["channels"], 1, 0,
                                            _ptr(s["field"]), 0, 8, bx, by, 1, _ptr(s["stats"]), st))
    return s["out"]


PATTERNS = [0x9966669999666699, 0x9669699669969669, 0xA55AA55A5AA55AA5, 0xAA55AA55AA55AA55,
            0xA55A5AA5A55A5AA5, 0x9966996666996699, 0xAA5555AA55AAAA55, 0x9669966996699669]


def _signs():
    """The eight patterns as +-1 over a cell's 64 pixels, row-major."""
    return torch.tensor([[1.0 if q >> i & 1 else -1.0 for i in range(64)] for q in PATTERNS], dtype=torch.float64,
                        device="cuda")


def _cells(plane):
    """The whole 8x8 cells of a plane, row-major: (cells, 64)."""
    H, W = plane.shape
    cy, cx = H // 8, W // 8
    return plane[:cy * 8, :cx * 8].reshape(cy, 8, cx, 8).permute(0, 2, 1, 3).reshape(cy * cx, 64)


def _grain_inputs(case, seed):
    """Two ring slots of a graded scene with film grain, the denoised frame, the pass's motion on
    the 8-pixel grid and eight earlier frames' grain history."""
    W, H, C = case["width"], case["height"], case["channels"]
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ys = torch.arange(H, device="cuda", dtype=torch.float32).unsqueeze(1)
    xs = torch.arange(W, device="cuda", dtype=torch.float32).unsqueeze(0)
    k = rng.uniform(0.0, 6.28, 4)
    # Large flat gradients, where grain is measured, with textured patches that fail the gates.
    clean = 0.45 + 0.22 * torch.sin(xs / 230.0 + k[0]) * torch.sin(ys / 190.0 + k[1])
    patch = (torch.sin(xs / 97.0 + k[2]) + torch.sin(ys / 71.0 + k[3]) > 1.2).to(torch.float32)
    clean = (clean + patch * 0.05 * torch.sin(xs / 1.7) * torch.sin(ys / 2.3)).contiguous()
    ring = torch.empty(2, H, W, C, device="cuda")
    for f in range(2):
        for c in range(C):
            g = torch.randn(1, 1, H + 2, W + 2, device="cuda", generator=gen)
            soft = torch.nn.functional.avg_pool2d(g, 3, stride=1)[0, 0]  # correlated over neighbours
            ring[f, :, :, c] = (clean + 0.012 * (0.5 * g[0, 0, 1:-1, 1:-1] + 1.5 * soft) * (0.6 + clean)).clamp(0, 1)
    denoised = clean.unsqueeze(2).expand(H, W, C).contiguous()
    bx, by = -(-W // 8), -(-H // 8)
    mv = torch.where(torch.rand(by, bx, 1, device="cuda", generator=gen) < 0.8,
                     torch.zeros(by, bx, 2, device="cuda", dtype=torch.int32),
                     torch.randint(-2, 3, (by, bx, 2), device="cuda", generator=gen, dtype=torch.int32)).contiguous()
    conf = torch.where(torch.rand(by, bx, device="cuda", generator=gen) < 0.9, 1.0, 0.4).contiguous()
    cells = (W // 8) * (H // 8)
    history = torch.zeros(9, cells, 9, device="cuda")
    signs = _signs().to(torch.float32)
    for slot in range(1, 9):
        noisy = clean + 0.012 * torch.randn(H, W, device="cuda", generator=gen)
        history[slot, :, :8] = (_cells(noisy).unsqueeze(1) * signs.unsqueeze(0)).sum(2)
        history[slot, :, 8] = (torch.rand(cells, device="cuda", generator=gen) < 0.8).to(torch.float32)
    lo, hi = 0.05 / 255.0, 32.0 / 255.0
    edges = torch.tensor([lo * (hi / lo) ** (i / 64) for i in range(65)], dtype=torch.float32, device="cuda")
    return ring.contiguous(), denoised, mv, conf, history, edges, bx, by, cells


def _grain_parts(hist, partials, records, history, persist):
    """The grain outputs by meaning, as views: lag sums apart from pixel counts and groups, the
    projections apart from the flat flags, the persistence sums apart from the cell counts."""
    part, rec, per = partials.view(-1, 48), records.view(16, 47), persist.view(8, 3)
    return {"hist": hist, "lags": part[:, :46], "counts": part[:, 46:], "record_lags": rec[:, :46],
            "record_counts": rec[:, 46], "projections": history[:, :, :8], "flags": history[:, :, 8],
            "persist_sums": per[:, 1:], "persist_counts": per[:, 0]}


def _prepare_grain(case, seed):
    W, H = case["width"], case["height"]
    lib = avd.load()
    ring, denoised, mv, conf, history, edges, bx, by, cells = _grain_inputs(case, seed)
    words = torch.tensor([w - (1 << 32) if w >= (1 << 31) else w for q in PATTERNS for w in (q & 0xFFFFFFFF, q >> 32)],
                         dtype=torch.int32, device="cuda")
    z = lambda *n, **k: torch.zeros(*n, device="cuda", **k)  # noqa: E731
    # hist, records and persist_record run on over a segment's frames, as a program keeps them.
    state = {"kind": "grain", "case": case, "lib": lib, "ring": ring, "denoised": denoised, "mv": mv, "conf": conf,
             "saved_mv": z(bx * by * 2, dtype=torch.int32), "saved_conf": z(bx * by), "words": words, "edges": edges,
             "history": history, "hist": z(2048, dtype=torch.int32), "partials": z(lib.avd_grain_partials_len(W, H)),
             "records": z(16 * 47), "persist_partials": z(lib.avd_grain_persist_partials_len(cells, 8)),
             "persist_record": z(24), "grid": (bx, by), "cells": cells}
    state["out"] = _grain_parts(state["hist"], state["partials"], state["records"], history, state["persist_record"])
    return state


def _run_grain(s):
    c, lib, st = s["case"], s["lib"], _stream()
    W, H, C, cells = c["width"], c["height"], c["channels"], s["cells"]
    bx, by = s["grid"]
    check(lib.avd_site_grain_save_vectors(_ptr(s["mv"]), _ptr(s["conf"]), _ptr(s["saved_mv"]), _ptr(s["saved_conf"]),
                                          0, 0, 0, bx * by, st))
    check(lib.avd_site_grain_measure(_ptr(s["ring"]), _ptr(s["denoised"]), W, H, C, 0, 0, 1, _ptr(s["saved_mv"]),
                                     _ptr(s["saved_conf"]), bx, by, 8, 0, 1, None, 0, 0, 1, _ptr(s["edges"]),
                                     _ptr(s["hist"]), _ptr(s["partials"]), st))
    check(lib.avd_site_grain_reduce(_ptr(s["partials"]), cells, _ptr(s["records"]), 0, st))
    check(lib.avd_site_grain_project(_ptr(s["ring"]), _ptr(s["denoised"]), _ptr(s["words"]), _ptr(s["history"]), W, H,
                                     C, 0, 0, 0, 1, st))
    check(lib.avd_site_grain_persist(_ptr(s["history"]), _ptr(s["persist_partials"]), _ptr(s["persist_record"]), 0, 0,
                                     cells, 8, st))
    return s["out"]


LAGS = [(0, dx) for dx in range(7)] + [(dy, dx) for dy in (1, 2, 3) for dx in range(-6, 7)]
AR_OFFSETS = [(dy, dx) for dy in (-3, -2, -1) for dx in range(-3, 4)] + [(0, dx) for dx in (-3, -2, -1)]


def _fit_inputs(case, seed):
    """Pooled records (46 lag sums and the pixel count) of grain of various softness."""
    rng = np.random.default_rng(seed)
    n = case["records"]
    rec = np.zeros((n, 47))
    for r in range(n):
        a, b, strength = rng.uniform(0.0, 0.6), rng.uniform(0.0, 0.6), rng.uniform(2e-5, 4e-4)
        pixels = float(rng.integers(60_000, 2_000_000))
        for k, (dy, dx) in enumerate(LAGS):
            white = rng.normal(0.0, 1.0 / math.sqrt(pixels)) if (dy, dx) != (0, 0) else 0.0
            rec[r, k] = pixels * strength * (a ** abs(dx) * b ** abs(dy) + white - (0.01 if (dy, dx) != (0, 0) else 0.0))
        rec[r, 46] = pixels
    return torch.from_numpy(rec).to("cuda")


def _prepare_fit(case, seed):
    n = case["records"]
    e = lambda *s, **k: torch.zeros(*s, device="cuda", **k)  # noqa: E731
    return {"kind": "grain_fit", "lib": avd.load(), "n": n, "records": _fit_inputs(case, seed),
            "corrected": e(n, 47, dtype=torch.float64), "weights": e(n, 24, dtype=torch.float64),
            "quantised": e(n, 24, dtype=torch.int32), "shifts": e(n, dtype=torch.int32),
            "solved": e(n, dtype=torch.int32)}


def _run_fit(s):
    check(s["lib"].avd_site_grain_fit(_ptr(s["records"]), s["n"], _ptr(s["corrected"]), _ptr(s["weights"]),
                                      _ptr(s["quantised"]), _ptr(s["shifts"]), _ptr(s["solved"]), _stream()))
    return {"corrected": s["corrected"][:, :46], "pixels": s["corrected"][:, 46],
            **{k: s[k] for k in ("weights", "quantised", "shifts", "solved")}}


# ---- the measured interface --------------------------------------------------------------------


def prepare(case, seed):
    return {"nlmeans": _prepare_stream, "nl4d": _prepare_stream, "host": _prepare_host, "noise": _prepare_noise,
            "grain": _prepare_grain, "grain_fit": _prepare_fit}[case["kind"]](case, seed)


def run(state):
    kind = state["kind"]
    if kind in ("nlmeans", "nl4d"):
        _emitted(state["engine"], state)
        return state["outs"]
    if kind == "host":
        den = state["engine"]
        den.push(state["frames"][state["at"] % CLIP_FRAMES])
        state["at"] += 1
        return [np.frombuffer(p, np.uint8) for p in den.recv()]
    return {"noise": _run_noise, "grain": _run_grain, "grain_fit": _run_fit}[kind](state)


def _sample_bytes(case):
    return 1 if case["depth"] == 8 else 2


def work(case):
    kind = case["kind"]
    if kind == "grain_fit":
        # Per record 20 rounds of 46 lags x 225 cell offsets (multiply, add) and the elimination.
        n = case["records"]
        return {"bytes": n * (2 * 47 + 24) * 8 + n * 26 * 4, "flops": n * (20 * 46 * 225 * 2 + 2 * 24 ** 3 / 3)}
    px = case["width"] * case["height"]
    if kind == "noise":
        C, blocks = case["channels"], -(-case["width"] // 16) * -(-case["height"] // 16)
        return {"bytes": 2 * px * C * 4 + blocks * (3 * C + 26) * 4 + 8, "flops": px * C * (12 + 8)}
    if kind == "grain":
        cells = (case["width"] // 8) * (case["height"] // 8)
        # Both slots and the denoised frame read, the partials and this frame's projections written,
        # eight earlier projections read; 46 lags x 64 products and 8 projections per cell.
        return {"bytes": cells * (3 * 64 + 48 + 9 + 8 * 9) * 4, "flops": cells * 64 * (46 * 2 + 8 + 20)}
    planes = _planes(case)
    total = sum(w * h for w, h in planes)
    nbytes = 2 * total * _sample_bytes(case)
    groups = [(planes[0], 1)] + ([(planes[1], 2)] if len(planes) > 1 else [])
    flops = 0.0
    for (w, h), C in groups:
        r = case["radius"]
        # Block motion on 16x16 blocks at step 8, radius 4: 3 operations per pixel and offset.  The
        # chroma pass refines the luma field (radius 1) instead of searching.
        motion = (w / 8.0) * (h / 8.0) * 81 * 256 * 3 * 2 * r * (1.25 if C == 1 else 9 / 81)
        if case["kind"] == "nl4d":
            refs = (w / case["step"]) * (h / case["step"])
            side, volumes = 2 * case["spatial"] + 1, case["group"] // (4 if r >= 2 else 2)
            flops += motion + refs * C * 192 * (side * side + volumes * 2 * r * 25)
            flops += refs * case["group"] * (C * (4096 + 576 + 256) + 64 * (C + 1))
        else:
            window = (2 * case["search"] + 1) ** 2
            flops += w * h * (window * (2 * r + 1) - 1) * (5 * C + 2 * (2 * case["patch"] + 1) + 7)
            flops += motion if case["motion"] else 0.0
    return {"bytes": float(nbytes), "flops": flops}


# ---- outputs in 64 bits ------------------------------------------------------------------------


def _exact_noise(case, seed):
    W, H, C = case["width"], case["height"], case["channels"]
    ring, field, bx, by = _noise_inputs(case, seed)
    f = ring.to(torch.float64)
    new, old = f[1], f[0]
    totals = torch.zeros(2, dtype=torch.float64, device="cuda")
    for c in range(C):
        p = new[:, :, c]
        m, u, d = p[1:-1], p[:-2], p[2:]
        resp = (4 * m[:, 1:-1] - 2 * (m[:, :-2] + m[:, 2:] + u[:, 1:-1] + d[:, 1:-1]) +
                u[:, :-2] + u[:, 2:] + d[:, :-2] + d[:, 2:])
        totals[c] = resp.abs().sum()
    nbx, nby = -(-W // 16), -(-H // 16)

    def blocks(p, fill=0.0):
        """(blocks, 256) of a plane, pixels past the frame holding `fill`."""
        full = torch.full((nby * 16, nbx * 16), fill, dtype=torch.float64, device="cuda")
        full[:H, :W] = p
        return full.view(nby, 16, nbx, 16).permute(0, 2, 1, 3).reshape(nby * nbx, 256)

    ys = torch.arange(H, device="cuda").unsqueeze(1).expand(H, W)
    xs = torch.arange(W, device="cuda").unsqueeze(0).expand(H, W)
    oy, ox = torch.meshgrid(torch.arange(nby, device="cuda") * 16, torch.arange(nbx, device="cuda") * 16, indexing="ij")
    oy, ox = oy.reshape(-1), ox.reshape(-1)
    bw, bh = (W - ox).clamp(max=16), (H - oy).clamp(max=16)
    moved = torch.zeros(nbx * nby, dtype=torch.float64, device="cuda")
    matched = torch.ones(nbx * nby, dtype=torch.bool, device="cuda")
    prev = old
    if field is not None:
        v = field.to(torch.int64)[(oy // 8).clamp(max=by - 1), (ox // 8).clamp(max=bx - 1)]
        up = lambda t: t.view(nby, nbx).repeat_interleave(16, 0).repeat_interleave(16, 1)[:H, :W]  # noqa: E731
        mx, my = xs + up(v[:, 0]), ys + up(v[:, 1])
        inside = (mx >= 0) & (mx < W) & (my >= 0) & (my < H)
        at = old[my.clamp(0, H - 1), mx.clamp(0, W - 1)]
        zr = blocks(new[:, :, 0] - old[:, :, 0])
        vr = blocks(torch.where(inside, new[:, :, 0] - at[:, :, 0], 0.0))
        left, top = ox + v[:, 0], oy + v[:, 1]
        span = (torch.minimum(left + bw, torch.tensor(W)) - left.clamp(min=0)).clamp(min=0) * \
            (torch.minimum(top + bh, torch.tensor(H)) - top.clamp(min=0)).clamp(min=0)
        px, safe = (bw * bh).double(), span.double().clamp(min=1)
        zvar = zr.square().sum(1) / px - (zr.sum(1) / px).square()
        vvar = vr.square().sum(1) / safe - (vr.sum(1) / safe).square()
        follows = ((v != 0).any(1)) & ((span == 0) | (vvar <= 0.5 * zvar))
        fits = (left >= 0) & (left + bw <= W) & (top >= 0) & (top + bh <= H)
        matched = ~(follows & ~fits)
        moved = (follows & fits).double()
        prev = torch.where(up(follows & fits).unsqueeze(2), at, old)
        valid = up(matched)
    else:
        valid = torch.ones(H, W, dtype=torch.bool, device="cuda")
    res = torch.where(valid.unsqueeze(2), new - prev, 0.0)
    inframe = blocks(valid.double()) > 0
    rec = torch.zeros(nbx * nby, 3 * C + 26, dtype=torch.float64, device="cuda")

    def texture(p):
        cells = blocks(torch.where(valid, p, 0.0)).view(-1, 4, 4, 4, 4).mean((2, 4))
        cols, rows = bw // 4, bh // 4
        i = torch.arange(4, device="cuda")
        okx, oky = i[None, :] < cols[:, None], i[None, :] < rows[:, None]
        right = (cells[:, :, :-1] - cells[:, :, 1:]).square() * (oky[:, :, None] & okx[:, None, 1:])
        down = (cells[:, :-1] - cells[:, 1:]).square() * (oky[:, 1:, None] & okx[:, None, :])
        pairs = rows * (cols - 1).clamp(min=0) + (rows - 1).clamp(min=0) * cols
        return torch.where(pairs > 0, (right.sum((1, 2)) + down.sum((1, 2))) / pairs.clamp(min=1), 0.0)

    for c in range(C):
        d = blocks(res[:, :, c])
        rec[:, c], rec[:, C + c] = d.sum(1), d.square().sum(1)
        rec[:, 2 * C + 1 if c == 0 else 2 * C + 26 + c] = texture(new[:, :, c])
    d = blocks(res[:, :, 0]).view(-1, 16, 16)
    rec[:, 2 * C] = (d[:, :, :-1] * d[:, :, 1:]).sum((1, 2))
    rec[:, 2 * C + 2] = moved
    n0 = torch.where(valid, new[:, :, 0], 0.0)
    mean = torch.where(valid, 0.5 * (new[:, :, 0] + prev[:, :, 0]), 0.0)
    quarter = lambda b: b.view(-1, 2, 8, 2, 8).permute(0, 1, 3, 2, 4).reshape(-1, 4, 64)  # noqa: E731
    q = torch.zeros(nbx * nby, 4, 6, dtype=torch.float64, device="cuda")
    qd, ql, qin = quarter(d.reshape(-1, 256)), quarter(blocks(n0)), quarter(inframe.double()) > 0
    q[:, :, 0], q[:, :, 1], q[:, :, 2] = qd.sum(2), qd.square().sum(2), ql.sum(2)
    grid = quarter(blocks(mean)).view(-1, 4, 4, 2, 4, 2).mean((3, 5))
    flat = (grid[:, :, :, :-1] - grid[:, :, :, 1:]).square().sum((2, 3)) + \
        (grid[:, :, :-1] - grid[:, :, 1:]).square().sum((2, 3))
    full = torch.stack([(bw >= 8 * (1 + (k & 1))) & (bh >= 8 * (1 + (k >> 1))) for k in range(4)], 1)
    q[:, :, 3] = torch.where(full, flat / 24.0, float(np.float32(3.0e38)))
    q[:, :, 4] = torch.where(qin, ql, float(np.float32(1e30))).amin(2)
    q[:, :, 5] = torch.where(qin, ql, float(np.float32(-1e30))).amax(2)
    q[~matched] = 0.0
    rec[:, 2 * C + 3:2 * C + 27] = q.view(-1, 24)
    return {"totals": totals, **_record_parts(rec.reshape(-1), C)}


def _exact_grain(case, seed):
    W, H, C = case["width"], case["height"], case["channels"]
    ring, denoised, mv, conf, history, edges, bx, by, cells = _grain_inputs(case, seed)
    cur, nxt, clean = ring[0, :, :, 0].double(), ring[1, :, :, 0].double(), denoised[:, :, 0].double()
    cx, cy = W // 8, H // 8
    ys = torch.arange(H, device="cuda").unsqueeze(1)
    xs = torch.arange(W, device="cuda").unsqueeze(0)
    v = mv.to(torch.int64)[(ys // 8).clamp(max=by - 1), (xs // 8).clamp(max=bx - 1)]
    moved = nxt[(ys + v[..., 1]).clamp(0, H - 1), (xs + v[..., 0]).clamp(0, W - 1)]
    g = (moved - cur) * float(np.float32(0.70710677))
    gc, cc, sc, mc = _cells(g), _cells(clean), _cells(cur), _cells(moved)
    total = gc.sum(1)
    std = ((gc.square().sum(1) - total.square() / 64) / 63).clamp(min=0).sqrt()
    mean, span = cc.mean(1), cc.amax(1) - cc.amin(1)
    iy, ix = torch.meshgrid(torch.arange(cy, device="cuda"), torch.arange(cx, device="cuda"), indexing="ij")
    interior = ((ix >= 1) & (ix + 2 <= cx) & (iy + 2 <= cy)).reshape(-1)
    usable = (span < 5 / 255) & (mean > 20 / 255) & (mean < 235 / 255) & \
        (torch.minimum(sc, mc).amin(1) >= 4 / 255) & (torch.maximum(sc, mc).amax(1) <= 251 / 255)
    trust = conf[:cy, :cx].reshape(-1) >= 0.8
    passes = usable & interior & trust & (std > 0.05 / 255)
    group = torch.where(passes, (torch.searchsorted(edges[1:64].double(), std, right=True) // 4).double(), 0.0)
    gm = total / 64
    pad = torch.nn.functional.pad(g[:cy * 8, :cx * 8], (6, 6, 0, 3))
    part = torch.zeros(cells, 48, dtype=torch.float64, device="cuda")
    for k, (dy, dx) in enumerate(LAGS):
        other = _cells(pad[dy:dy + cy * 8, 6 + dx:6 + dx + cx * 8])
        part[:, k] = ((gc - gm[:, None]) * (other - gm[:, None])).sum(1)
    part[:, 46] = 64.0
    part[~passes] = 0.0
    part[:, 47] = group
    records = torch.zeros(16, 47, dtype=torch.float64, device="cuda")
    records.index_add_(0, group.long().clamp(max=15), part[:, :47])
    hist = history.double()
    hist[0, :, :8] = (sc.unsqueeze(1) * _signs().unsqueeze(0)).sum(2)
    hist[0, :, 8] = ((span < 5 / 255) & (mean > 20 / 255) & (mean < 235 / 255) & (sc.amin(1) >= 4 / 255) &
                     (sc.amax(1) <= 251 / 255)).double()
    persist = torch.zeros(8, 3, dtype=torch.float64, device="cuda")
    for lag in range(8):
        ear = hist[8 - lag]
        both = (hist[0, :, 8] * ear[:, 8]) > 0.5
        a, b = hist[0, both, :8], ear[both, :8]
        persist[lag, 0] = both.sum()
        persist[lag, 1] = (a.square() + b.square()).sum() / 1024
        persist[lag, 2] = (a * b).sum() / 512
    return _grain_parts(None, part, records, hist, persist)


def _exact_fit(case, seed):
    rec = _fit_inputs(case, seed).cpu().numpy().astype(np.longdouble)
    index = {lag: k for k, lag in enumerate(LAGS)}

    def lane(dy, dx):
        return index.get((-dy, -dx) if dy < 0 or (dy == 0 and dx < 0) else (dy, dx))

    term = np.zeros((46, 46), dtype=np.longdouble)  # the cell-mean term of each lag is linear in the record
    for k, (dy, dx) in enumerate(LAGS):
        for oy in range(-7, 8):
            for ox in range(-7, 8):
                j = lane(dy + oy, dx + ox)
                if j is not None:
                    term[k, j] += np.longdouble((8 - abs(oy)) * (8 - abs(ox))) / 4096
    corrected, weights = np.zeros((len(rec), 47)), np.zeros((len(rec), 24))
    for r, row in enumerate(rec):
        measured = row[:46] / row[0]
        rho = measured.copy()
        for _ in range(20):
            t = term @ rho
            rho = measured * (1 - t[0]) + t
        lags = rho * row[0]
        corrected[r, :46], corrected[r, 46] = lags, row[46]
        m = np.array([[lags[lane(a[0] - b[0], a[1] - b[1])] for b in AR_OFFSETS] for a in AR_OFFSETS]) / row[46]
        y = np.array([lags[lane(*a)] for a in AR_OFFSETS]) / row[46]
        for c in range(24):  # elimination with partial pivoting, in extended precision
            p = c + int(np.argmax(np.abs(m[c:, c])))
            m[[c, p]], y[[c, p]] = m[[p, c]], y[[p, c]]
            for i in range(c + 1, 24):
                f = m[i, c] / m[c, c]
                m[i] -= f * m[c]
                y[i] -= f * y[c]
        w = np.zeros(24, dtype=np.longdouble)
        for i in range(23, -1, -1):
            w[i] = (y[i] - (m[i, i + 1:] * w[i + 1:]).sum()) / m[i, i]
        weights[r] = w
    return {"corrected": corrected[:, :46], "pixels": corrected[:, 46], "weights": weights, "quantised": None, "shifts": None, "solved": None}


def exact(case, seed):
    """The outputs in 64 bits; None for frames, whose outputs are whole sample codes."""
    fn = {"noise": _exact_noise, "grain": _exact_grain, "grain_fit": _exact_fit}.get(case["kind"])
    return fn(case, seed) if fn else None

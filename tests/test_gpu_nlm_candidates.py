"""Every candidate the launch tuner may choose for an NLM frame, in both forms, at shapes where tiles end
in the frame's last rows and columns, on both sides of the plane size that splits the offsets: the candidates
give the same bits, and those are the FP64 oracle's frame; and the tuner, which compares them on its own
content at an engine's construction, drops none."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import avd
from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, ptr, require_gpu

pytestmark = pytest.mark.gpu


def _pointers(tensors):
    return (ctypes.c_void_p * max(len(tensors), 1))(*(ptr(t) for t in tensors))


@pytest.mark.parametrize("W,H,C,P,S,pairs,conf", [
    (1, 1, 1, 4, 2, 1, True), (33, 60, 1, 2, 3, 2, False), (31, 61, 1, 2, 8, 1, True), (32, 59, 2, 2, 3, 2, True),
    (17, 65, 2, 0, 1, 0, False), (40, 121, 1, 0, 2, 1, False), (19, 62, 1, 1, 4, 3, True), (16, 117, 2, 3, 0, 1, True),
    (35, 57, 1, 4, 4, 0, False), (64, 55, 2, 5, 2, 1, False), (9, 53, 1, 6, 5, 1, True), (65, 51, 2, 7, 1, 2, True),
    (33, 49, 1, 8, 8, 1, False), (15, 97, 2, 8, 8, 1, True), (1031, 1019, 1, 1, 1, 1, True), (1025, 1023, 2, 1, 1, 1, True)])
def test_candidates_give_the_same_bits(W, H, C, P, S, pairs, conf):
    require_gpu()
    print(f"candidates {W}x{H} C {C} P {P} S {S} pairs {pairs} conf {conf}", flush=True)
    rng = np.random.default_rng(W * 3 + H + C)
    h2, off, self_weight = float(O.h2_inv_norm(1.2, P)), 0.002, 0.8
    spread = min(np.sqrt(2.0 * (1.0 / h2 + off)) / (2 * P + 1), 1.0)
    frames = [rng.uniform(0.5 - spread / 2, 0.5 + spread / 2, W * H * C).astype(np.float32) for _ in range(2 * pairs + 1)]
    bx, by = -(-W // 8), -(-H // 8)
    confs = [rng.uniform(0.2, 1, bx * by).astype(np.float32) for _ in range(2 * pairs)]
    lut = O.spatial_offset_lut(S, off)
    sums = [np.zeros(W * H * C), np.zeros(W * H), np.zeros(W * H)]
    for k in range(pairs):
        cf, cb = (confs[2 * k], confs[2 * k + 1]) if conf else (None, None)
        O.nlm_pair(frames[0], frames[1 + 2 * k], frames[2 + 2 * k], W, H, C, P, S, h2, off, cf, cb, 8, bx, by, *sums,
                   precision="f64")
    O.nlm_single(frames[0], W, H, C, P, S, h2, lut, *sums, precision="f64")
    want = O.nlm_finish(frames[0], *sums, self_weight, W * H, C, "f64")
    w = L.NlmWindow()
    w.width, w.height, w.channels, w.patch_radius, w.search_radius = W, H, C, P, S
    w.h2_inv_norm, w.noise_offset, w.step, w.blocks_x, w.blocks_y = h2, off, 8, bx, by
    f, c, d_lut = [dev(x) for x in frames], [dev(x) for x in confs], dev(lut)
    fwd, bwd, cf, cb = (_pointers(x) for x in (f[1::2], f[2::2], c[0::2], c[1::2]))
    first = None
    for form, candidates in ((0, 3), (1, 2)):
        for candidate in range(candidates):
            acc, out = [torch.full((n,), 77.0, device="cuda") for n in (W * H * C, W * H, W * H)], torch.zeros(W * H * C, device="cuda")
            L.check(avd.load().avd_nlm_frame_for_test(
                ctypes.byref(w), form, candidate, pairs, ptr(f[0]), fwd, bwd, cf if conf else None, cb if conf else None,
                ptr(d_lut), self_weight, ptr(acc[0]), ptr(acc[1]), ptr(acc[2]), ptr(out), None))
            got = host(out)
            if first is None:
                first = got
                # exp2 of a rounded distance: up to about 1e-4 of a weight, as in the windows' other tests
                assert np.allclose(got, want, rtol=1e-4, atol=1e-6), np.max(np.abs(got - want))
            assert np.array_equal(got.view(np.uint32), first.view(np.uint32)), (form, candidate)


@pytest.mark.parametrize("chroma,W,H,P,S,r,hq", [("gray", 67, 59, 2, 7, 0, False), ("444", 61, 71, 8, 8, 1, False),
                                                 ("420", 131, 117, 4, 2, 2, True), ("422", 90, 53, 6, 3, 1, True),
                                                 ("gray", 70, 65, 0, 1, 3, False)])
def test_the_tuner_drops_none(chroma, W, H, P, S, r, hq):
    require_gpu()
    print(f"tuner {chroma} {W}x{H} P {P} S {S} r {r} hq {hq}", flush=True)
    layout = {"gray": 0, "420": 1, "422": 2, "444": 3}[chroma]
    geom = L.Geometry(W, H, layout, L.SampleFormat.u16(10), L.SampleFormat.u16(10), 0)
    opts = avd.nlmeans_options(temporal=1 if r else 0, temporal_radius=r, patch_radius=P, search_radius=S,
                               hq=1 if hq else 0, **({"sigma": 0.01} if hq else {"strength": 1.2}))
    avd.set_tuning(True)
    avd.build_engine("nlmeans", geom, luma=opts, chroma=opts if layout else None)
    entries = [e for e in avd.tuning_entries() if f"P{P} S{S} {W}x{H}" in e["key"]]
    assert {e["site"] for e in entries} == {"nlm_single", "nlm_window"} | ({"nlm_pair"} if r else set())
    for e in entries:
        assert len(e["ms"]) == (2 if e["site"] == "nlm_window" else 3) and all(t >= 0 for t in e["ms"]), e


def test_the_tuner_times_the_launches_a_frame_makes():
    """A spatial pass's only window starts and finishes the frame, and a radius-1 pass's only pair starts
    the sums: they are sites of their own, not those of passes with more windows."""
    require_gpu()
    W, H = 83, 47
    geom = L.Geometry(W, H, 0, L.SampleFormat.u8(), L.SampleFormat.u8(), 0)
    avd.set_tuning(True)
    sites = {}
    for r in (2, 1, 0):
        opts = avd.nlmeans_options(temporal=1 if r else 0, temporal_radius=r, patch_radius=2, search_radius=2)
        avd.build_engine("nlmeans", geom, luma=opts)
        sites[r] = {(e["site"], e["key"]) for e in avd.tuning_entries() if f"{W}x{H}" in e["key"]}
    assert {s for s, _ in sites[1] - sites[2]} == {"nlm_pair", "nlm_window"}
    assert {s for s, _ in sites[0] - sites[1]} == {"nlm_single", "nlm_window"}

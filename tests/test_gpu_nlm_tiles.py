"""NLM windows at the edges of their tiles against the FP64 oracle: frames one pixel around a tile of
64 - 2P rows, of one pixel, and on both sides of the plane size that splits the offsets over waves;
every patch radius, search radii 0 to 8, one and two channels; then the same frames finished by the
engine's fused launches in both forms."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import avd
from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, ptr, require_gpu, run_engine, words_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,C,P,S", [
    (1, 1, 1, 4, 2), (33, 60, 1, 2, 3), (31, 61, 1, 2, 8), (32, 59, 2, 2, 3), (17, 65, 2, 0, 1), (40, 121, 1, 0, 2),
    (19, 62, 1, 1, 4), (16, 117, 2, 3, 0), (35, 57, 1, 4, 4), (64, 55, 2, 5, 2), (9, 53, 1, 6, 5), (65, 51, 2, 7, 1),
    (33, 49, 1, 8, 8), (15, 97, 2, 8, 8), (1031, 1019, 1, 1, 1), (1025, 1023, 2, 1, 1)])
def test_windows_match_the_oracle(W, H, C, P, S):
    require_gpu()
    print(f"windows {W}x{H} C {C} P {P} S {S}", flush=True)
    rng = np.random.default_rng(W * 3 + H + C)
    frames = [rng.uniform(0, 1, W * H * C).astype(np.float32) for _ in range(3)]
    h2, off = float(O.h2_inv_norm(1.2, P)), 0.01
    lut = O.spatial_offset_lut(S, off)
    bx, by = -(-W // 8), -(-H // 8)
    conf = [rng.uniform(0, 1, bx * by).astype(np.float32) for _ in range(2)]
    want = [np.zeros(W * H * C), np.zeros(W * H), np.zeros(W * H)]
    O.nlm_pair(frames[0], frames[1], frames[2], W, H, C, P, S, h2, off, conf[0], conf[1], 8, bx, by, *want,
               precision="f64")
    O.nlm_single(frames[0], W, H, C, P, S, h2, lut, *want, precision="f64")
    w = L.NlmWindow()
    w.width, w.height, w.channels, w.patch_radius, w.search_radius = W, H, C, P, S
    w.h2_inv_norm, w.noise_offset, w.step, w.blocks_x, w.blocks_y = h2, off, 8, bx, by
    got = [torch.zeros(W * H * C, device="cuda"), torch.zeros(W * H, device="cuda"), torch.zeros(W * H, device="cuda")]
    f, c, d_lut = [dev(x) for x in frames], [dev(x) for x in conf], dev(lut)
    L.check(avd.load().avd_site_nlm_pair(ctypes.byref(w), ptr(f[0]), ptr(f[1]), ptr(f[2]), ptr(c[0]), ptr(c[1]),
                                         ptr(got[0]), ptr(got[1]), ptr(got[2]), None))
    L.check(avd.load().avd_site_nlm_single(ctypes.byref(w), ptr(f[0]), ptr(d_lut), ptr(got[0]), ptr(got[1]),
                                           ptr(got[2]), None))
    for g, t in zip((host(x) for x in got), want):
        # exp2 of a rounded distance: up to about 1e-4 of a weight, as in the windows' other tests
        assert np.allclose(g, t, rtol=1e-4, atol=1e-6), np.max(np.abs(g - t))


@pytest.mark.parametrize("r", [0, 1, 3])
def test_engine_forms_agree_at_a_tile_edge(r):
    require_gpu()
    W, H, depth, frames = 66, 57, 10, 4
    clip = avd.synth.clip(frames, W, H, depth, 21 + r, chroma="420", sigma_luma=12.0, sigma_chroma=8.0)
    geom = L.Geometry(W, H, 1, L.SampleFormat.u16(depth), L.SampleFormat.u16(depth), 0)
    opts = avd.nlmeans_options(temporal=1 if r else 0, temporal_radius=r, patch_radius=4, search_radius=3)
    spec = O.NlmSpec(r, 3, 4, 1.2, 1.0)
    outs = {}
    for form in ("plain", "batched"):
        eng = avd.build_engine("nlmeans", geom, luma=opts, chroma=opts)
        eng.set_nlm_form(form)
        outs[form] = run_engine(eng, [[words_dev(p.numpy(), depth) for p in f] for f in clip], depth, avd.plane_dims(geom))
    luma, _ = O.run_stream(O.NlmPass(spec, W, H, 1, depth, depth), [[O.pack_plane(f[0].numpy(), depth)] for f in clip])
    for t in range(frames):
        for a, b in zip(outs["plain"][t], outs["batched"][t]):
            assert np.array_equal(a, b)
        got = O.unpack_plane(outs["plain"][t][0], depth, W * H).astype(int)
        assert np.abs(got - O.unpack_plane(luma[t][0], depth, W * H).astype(int)).max() <= 1

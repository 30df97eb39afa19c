"""NLM windows of frames past the tile rows that 16 bits of a grid hold: the rows of a tall frame are those
of its lower part alone, away from where that part begins."""
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


@pytest.mark.parametrize("H,C,P", [(48 * (1 << 16) + 5, 1, 8), (54 * (1 << 16) + 1, 2, 5)])
def test_tall_frames(H, C, P):
    require_gpu()
    print(f"tall {H} rows C {C} P {P}", flush=True)
    part, S = (1 << 20) + 300, 1  # both past the plane size that splits the offsets
    rng = np.random.default_rng(H + C)
    h2 = float(O.h2_inv_norm(1.2, P))
    frames = [dev((0.5 + 0.02 * rng.random(H * C)).astype(np.float32)) for _ in range(3)]
    lut = dev(O.spatial_offset_lut(S, 0.001))
    outs = {}
    for rows in (H, part):
        w = L.NlmWindow()
        w.width, w.height, w.channels, w.patch_radius, w.search_radius = 1, rows, C, P, S
        w.h2_inv_norm, w.noise_offset, w.step, w.blocks_x, w.blocks_y = h2, 0.001, 1, 1, 1
        f = [x[(H - rows) * C:].contiguous() for x in frames]
        fwd, bwd = ((ctypes.c_void_p * 1)(ptr(x)) for x in f[1:])
        for form in (0, 1):
            sums = [torch.zeros(n, device="cuda") for n in (rows * C, rows, rows)]
            out = torch.full((rows * C,), -7.0, device="cuda")
            L.check(avd.load().avd_nlm_frame_for_test(ctypes.byref(w), form, 0, 1, ptr(f[0]), fwd, bwd, None, None, ptr(lut),
                                                      1.0, ptr(sums[0]), ptr(sums[1]), ptr(sums[2]), ptr(out), None))
            outs[rows, form] = host(out).view(np.uint32).reshape(rows, C)
    for form in (0, 1):
        assert np.array_equal(outs[H, form], outs[H, 0])
        assert np.array_equal(outs[H, form][H - part + P + S:], outs[part, form][P + S:])
        # The rows above it are finished too (a frame of half-codes, every output of which lies in its range).
        assert outs[H, form].view(np.float32).min() >= 0.49

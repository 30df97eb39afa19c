"""The temporal records of frames on both sides of the block counts where a workgroup stops taking a
block of its own (1024 blocks, 1280 with motion), against the oracle, bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("luma", [True, False])
@pytest.mark.parametrize("w,h,c", [(512, 512, 1), (511, 500, 2), (400, 656, 1), (393, 641, 2), (640, 512, 1), (633, 505, 2),
                                   (16, 1281 * 16, 1), (672, 488, 2)])
def test_both_sides_of_the_line(w, h, c, luma):
    require_gpu()
    print(f"temporal {w}x{h} C {c} luma {luma}", flush=True)
    rng = np.random.default_rng(w + h + c)
    ring = rng.uniform(0.0, 1.0, (2, h, w, c)).astype(np.float32)
    bx, by = -(-w // 8), -(-h // 8)
    field = rng.integers(-6, 7, (by, bx, 2)).astype(np.int32)
    field[rng.random((by, bx)) < 0.3] = 0
    ring[0, :, 2:] = np.where(rng.random((h, w - 2, c)) < 0.5, ring[1, :, :-2], ring[0, :, 2:])  # some blocks follow
    field[rng.random((by, bx)) < 0.3] = (2, 0)
    d_ring, d_mv = dev(ring), dev(field)
    for motion in (None, (field.reshape(-1), 0, 8, bx, by)):
        stats = torch.full((O.temporal_slot_len(w, h, c),), -7.0, device="cuda")
        L.check(L.load().avd_site_noise_temporal_stats(
            ctypes.c_void_p(d_ring.data_ptr()), w, h, c, 1, 0,
            None if motion is None else ctypes.c_void_p(d_mv.data_ptr()), 0, 8, bx, by, 1 if luma else 0,
            ctypes.c_void_p(stats.data_ptr()), None))
        want = O.temporal_stats(ring, w, h, c, 1, 0, luma, motion)
        assert np.array_equal(host(stats).view(np.uint32), want.view(np.uint32))

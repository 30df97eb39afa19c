"""The radius-0 block match (a block's SAD and confidence where its seed stands) against the oracle:
ragged frames down to less than a block, one and two channels, more neighbours than one round holds,
seeds that leave the frame on every side."""
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


@pytest.mark.parametrize("W,H,C,neighbours,ov", [(80, 56, 1, 4, 8), (77, 43, 2, 1, 8), (13, 9, 1, 5, 8), (3, 2, 2, 2, 8),
                                                 (16, 16, 2, 16, 8), (131, 67, 1, 9, 12), (47, 33, 1, 3, 0)])
def test_radius_zero_matches_the_oracle(W, H, C, neighbours, ov):
    require_gpu()
    print(f"radius 0 {W}x{H} C {C} neighbours {neighbours}", flush=True)
    rng = np.random.default_rng(W * 31 + H + C)
    ring = rng.integers(0, 4096, (neighbours + 1, H, W, C)).astype(np.uint16)
    g = O.MotionGeom(W, H, 16, ov, 0, 1)
    centre = neighbours // 2
    slots = [i for i in range(neighbours + 1) if i != centre]
    seeds = rng.integers(-40, 41, (neighbours, g.blocks, 2)).astype(np.int32)
    seeds[:, ::3] = 0
    mp = L.MotionPass()
    mp.width, mp.height, mp.channels, mp.blksize, mp.overlap = W, H, C, 16, ov
    mp.search_radius, mp.pyramid_levels, mp.centre_slot, mp.neighbours = 0, 1, centre, neighbours
    mp.max_value, mp.sad_floor, mp.thsad = 4095.0, 3.0, 90.0
    mv = torch.full((neighbours * g.blocks * 2,), 999, dtype=torch.int32, device="cuda")
    conf = torch.full((neighbours * g.blocks,), -1.0, device="cuda")
    d_ring, ns, d_seeds = dev(ring.view(np.int16)), dev(np.asarray(slots, np.int32)), dev(seeds)
    for given in (d_seeds, None):  # around seeds, then where the blocks stand
        if given is None:
            L.check(avd.load().avd_site_motion(ctypes.byref(mp), ptr(d_ring), ptr(ns), ptr(mv), ptr(conf), None))
        else:
            L.check(avd.load().avd_site_motion_refine(ctypes.byref(mp), ptr(d_ring), ptr(ns), ptr(given), 0, ptr(mv),
                                                      ptr(conf), None))
        got_mv, got_conf = host(mv).reshape(neighbours, -1), host(conf).reshape(neighbours, -1)
        lane0 = [np.ascontiguousarray(f[..., 0].reshape(-1).astype(np.int32)) for f in ring]
        for i, s in enumerate(slots):
            want = seeds[i].reshape(-1) if given is not None else np.zeros(g.blocks * 2, np.int32)
            want_mv, want_conf = O.motion_refine(g, [lane0[centre]], [lane0[s]], want, 4095.0, 3.0, 90.0, radius=0)
            assert np.array_equal(got_mv[i], want_mv)
            assert np.array_equal(got_conf[i], want_conf)

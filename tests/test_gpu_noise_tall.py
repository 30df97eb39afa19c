"""Spatial noise totals of frames taller than one grid layer of workgroups (2^19 rows), and than the
16 bits of a grid's y extent (2^20 rows at sixteen a workgroup), against the oracle."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,c", [(3, (1 << 19) + 1, 1), (4, (1 << 20) + 37, 1), (3, (1 << 20) + 16, 2)])
def test_tall_frames(w, h, c):
    require_gpu()
    print(f"tall {w}x{h} C {c}", flush=True)
    ring = np.random.default_rng(h + c).uniform(0.0, 1.0, (1, h, w, c)).astype(np.float32)
    n = O.noise_partials_len(w, h)
    d_ring = dev(ring)
    partials, results = torch.full((n,), -7.0, device="cuda"), torch.full((2,), -7.0, device="cuda")
    L.check(L.load().avd_site_noise_spatial(ctypes.c_void_p(d_ring.data_ptr()), w, h, c, 0,
                                            ctypes.c_void_p(partials.data_ptr()), ctypes.c_void_p(results.data_ptr()),
                                            0, None))
    want = O.noise_partial(ring, w, h, c, 0)
    assert np.array_equal(host(partials).view(np.uint32), want.view(np.uint32))
    assert np.array_equal(host(results).view(np.uint32), O.noise_reduce(want)[:2].view(np.uint32))

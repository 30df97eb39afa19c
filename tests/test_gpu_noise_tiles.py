"""The noise kernels at the edges of their workgroups against the oracle, bit for bit: block counts
around the sixteen planes a workgroup holds, tile counts around its sixteen tile sums and around the
reduce's batches, frames below a block, a tile or the mask, one and two channels, and samples that are
not finite."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu


def _frames(w, h, c, seed, odd_values):
    rng = np.random.default_rng(seed)
    ring = rng.uniform(0.0, 1.0, (2, h, w, c)).astype(np.float32)
    if odd_values:
        for v in (np.nan, np.inf, -np.inf, -0.0, 3.0e38):
            ring[rng.integers(2), rng.integers(h), rng.integers(w), rng.integers(c)] = v
    return ring


def _same(got, want, what):
    # NaN payloads are the operation order's; every other value matches in its bits.
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    ok = ~np.isnan(want)
    bad = np.flatnonzero(got[ok].view(np.uint32) != want[ok].view(np.uint32))
    assert bad.size == 0, (what, bad[:8], got[ok][bad[:8]], want[ok][bad[:8]])


@pytest.mark.parametrize("odd_values", [False, True])
@pytest.mark.parametrize("w,h,c", [(256, 16, 1), (255, 17, 1), (272, 31, 1), (15, 255, 1), (128, 16, 2), (129, 33, 2),
                                   (8, 8, 1), (9, 7, 2), (16, 1, 1), (3, 300, 2), (241, 65, 1)])
def test_temporal_records(w, h, c, odd_values):
    require_gpu()
    print(f"temporal {w}x{h} C {c}", flush=True)
    ring = _frames(w, h, c, w + 7 * h + c, odd_values)
    rng = np.random.default_rng(w)
    bx, by = -(-w // 8), -(-h // 8)
    field = rng.integers(-6, 7, (by, bx, 2)).astype(np.int32)
    field[rng.random((by, bx)) < 0.3] = 0
    field[rng.random((by, bx)) < 0.1] = (2**31 - 1, -2**31)
    d_ring, d_mv = dev(ring), dev(field)
    for motion in (None, (field.reshape(-1), 0, 8, bx, by)):
        for luma in (True, False):
            stats = torch.full((O.temporal_slot_len(w, h, c),), -7.0, device="cuda")
            L.check(L.load().avd_site_noise_temporal_stats(
                ctypes.c_void_p(d_ring.data_ptr()), w, h, c, 1, 0,
                None if motion is None else ctypes.c_void_p(d_mv.data_ptr()), 0, 8, bx, by, 1 if luma else 0,
                ctypes.c_void_p(stats.data_ptr()), None))
            with np.errstate(all="ignore"):
                want = O.temporal_stats(ring, w, h, c, 1, 0, luma, motion)
            _same(host(stats), want, (motion is not None, luma))


@pytest.mark.parametrize("odd_values", [False, True])
@pytest.mark.parametrize("w,h,c", [(256, 16, 1), (257, 17, 1), (128, 16, 2), (129, 15, 2), (31, 9, 1), (2, 2, 1), (1, 40, 2),
                                   (3, 3, 2), (32, 2048, 1), (96, 2055, 1), (2048, 513, 1), (1280, 1601, 1)])
def test_spatial_totals(w, h, c, odd_values):
    require_gpu()
    print(f"spatial {w}x{h} C {c}", flush=True)
    ring = _frames(w, h, c, w + 3 * h + c, odd_values)
    n = O.noise_partials_len(w, h)
    d_ring = dev(ring)
    partials, results = torch.full((n + 1,), -7.0, device="cuda"), torch.full((6,), -7.0, device="cuda")
    with np.errstate(all="ignore"):
        want_p = O.noise_partial(ring, w, h, c, 1)
        want_r = O.noise_reduce(want_p)
    for at in (0, 1):  # the caller's floats, eight-byte aligned or not
        L.check(L.load().avd_site_noise_spatial(ctypes.c_void_p(d_ring.data_ptr()), w, h, c, 1,
                                                ctypes.c_void_p(partials[at:].data_ptr()),
                                                ctypes.c_void_p(results.data_ptr()), 2, None))
        _same(host(partials)[at:at + n], want_p, "partials")
        _same(host(results)[4:], want_r[:2], "totals")

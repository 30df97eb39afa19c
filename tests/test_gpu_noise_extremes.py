"""The temporal records' quarter extremes over values a picture does not hold: quarters of NaN alone, of
infinities, of values past +-1e30 (what a pixel outside the frame counts as), with and without pixels
outside the frame, against the oracle; and a signalling NaN, which counts as any NaN."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu


def _records(ring, w, h, c, field):
    bx, by = -(-w // 8), -(-h // 8)
    stats = torch.full((O.temporal_slot_len(w, h, c),), -7.0, device="cuda")
    d_ring, d_mv = dev(ring), None if field is None else dev(field)
    L.check(L.load().avd_site_noise_temporal_stats(
        ctypes.c_void_p(d_ring.data_ptr()), w, h, c, 1, 0, None if field is None else ctypes.c_void_p(d_mv.data_ptr()),
        0, 8, bx, by, 1, ctypes.c_void_p(stats.data_ptr()), None))
    return host(stats).reshape(-1, 3 * c + 26)


def _extremes(records, c):
    return records[:, 2 * c + 3:2 * c + 27].reshape(-1, 4, 6)[:, :, 4:]


# The larger frames take more workgroups than a small one has blocks.
SIZES = [(64, 32, 1), (61, 27, 1), (48, 40, 2), (640, 640, 1), (635, 637, 2)]


@pytest.mark.parametrize("motion", [False, True])
@pytest.mark.parametrize("w,h,c", SIZES)
def test_extremes_of_unusual_quarters(w, h, c, motion):
    require_gpu()
    print(f"extremes {w}x{h} C {c} motion {motion}", flush=True)
    rng = np.random.default_rng(w + h + c)
    ring = rng.uniform(0.0, 1.0, (2, h, w, c)).astype(np.float32)
    values = [np.nan, np.inf, -np.inf, 5.0e30, -5.0e30]
    for k, (y, x) in enumerate((y, x) for y in range(0, h, 8) for x in range(0, w, 8)):
        if k % 3 == 0:
            ring[1, y:y + 8, x:x + 8] = values[k // 3 % len(values)]
    field = np.zeros((-(-h // 8), -(-w // 8), 2), np.int32) if motion else None
    mv = (field.reshape(-1), 0, 8, field.shape[1], field.shape[0]) if motion else None
    with np.errstate(all="ignore"):
        want = _extremes(O.temporal_stats(ring, w, h, c, 1, 0, True, mv).reshape(-1, 3 * c + 26), c)
    got = _extremes(_records(ring, w, h, c, field), c)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))


@pytest.mark.parametrize("w,h,c", SIZES)
def test_a_signalling_nan_counts_as_any(w, h, c):
    require_gpu()
    print(f"signalling NaN {w}x{h} C {c}", flush=True)
    rng = np.random.default_rng(w * h + c)
    ring = rng.uniform(0.0, 1.0, (2, h, w, c)).astype(np.float32)
    at = rng.random((h, w)) < 0.1
    extremes = []
    for nan in (0x7FC00001, 0x7F800001):  # quiet, signalling
        ring.view(np.uint32)[1, :, :, 0][at] = nan
        extremes.append(_extremes(_records(ring, w, h, c, None), c))
    assert not np.isnan(extremes[0]).any()
    assert np.array_equal(extremes[0].view(np.uint32), extremes[1].view(np.uint32))

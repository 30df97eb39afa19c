"""The grain kernels at the edges of their workgroups against the oracle, bit for bit: cell grids around
the 16 x 2 cells a measuring group holds and the 8 x 4 a projecting one does, frames with part cells and
without interior ones, one to four channels, vectors that leave the frame, samples that are not finite,
and partials off the vector load's alignment around the reduce's batches."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from avd import _lib as L

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu

SIZES = [(8, 8, 1, 0), (128, 16, 1, 0), (136, 24, 1, 0), (143, 23, 2, 1), (127, 47, 3, 2), (264, 40, 4, 3), (24, 16, 1, 0),
         (16, 200, 1, 0), (71, 72, 1, 0)]


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _same(got, want, what):
    # NaN payloads are the operation order's; every other value matches in its bits.
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    ok = ~np.isnan(want)
    bad = np.flatnonzero(got[ok].view(np.uint32) != want[ok].view(np.uint32))
    assert bad.size == 0, (what, bad[:8], got[ok][bad[:8]], want[ok][bad[:8]])


def _scene(w, h, c, ch, odd_values):
    rng = np.random.default_rng(w * 7 + h + c)
    ring = rng.uniform(0, 1, (2, h, w, c)).astype(np.float32)
    ring[..., ch] = 0.4 + 0.004 * rng.standard_normal((2, h, w))
    den = rng.uniform(0, 1, (h, w, c)).astype(np.float32)
    den[..., ch] = 0.4 + np.linspace(0, 0.01, w)
    if odd_values:
        for v in (np.nan, np.inf, -np.inf, -0.0, 3.0e38):
            ring[rng.integers(2), rng.integers(h), rng.integers(w), ch] = v
        den[rng.integers(h), rng.integers(w), ch] = np.nan
    return rng, ring, den


@pytest.mark.parametrize("odd_values", [False, True])
@pytest.mark.parametrize("w,h,c,ch", SIZES)
def test_measure(w, h, c, ch, odd_values):
    require_gpu()
    print(f"measure {w}x{h} C {c}", flush=True)
    rng, ring, den = _scene(w, h, c, ch, odd_values)
    cells = (w // 8) * (h // 8)
    for step, has_source in ((8, 1), (12, 1), (8, 0)):
        bx, by = -(-w // step), max(1, h // step - 1)  # a grid short of the frame: the last row's vectors go on
        mv = rng.integers(-3, 4, (by * bx, 2)).astype(np.int32)
        mv[rng.random(by * bx) < 0.5] = 0
        mv[rng.random(by * bx) < 0.1] = (-70000, 70000)
        conf = np.where(rng.random(by * bx) < 0.1, 0.79, 0.8).astype(np.float32)
        hist = torch.full((2048,), 5, dtype=torch.int32, device="cuda")
        part = torch.full((cells * 48,), -7.0, device="cuda")
        d = [dev(a) for a in (ring, den, mv.reshape(-1), conf, O.grain_bucket_edges())]
        L.check(L.load().avd_site_grain_measure(_p(d[0]), _p(d[1]), w, h, c, ch, 0, 1, _p(d[2]), _p(d[3]), bx, by, step,
                                                0, has_source, None, 0, 0, 1, _p(d[4]), _p(hist), _p(part), None))
        with np.errstate(all="ignore"):
            want_hist, want_part = O.grain_measure(ring, den, w, h, c, ch, 0, 1, mv.reshape(-1), conf, bx, by, step,
                                                   has_source=bool(has_source))
        assert np.array_equal(host(hist), want_hist + 5), step
        _same(host(part), want_part, step)


@pytest.mark.parametrize("odd_values", [False, True])
@pytest.mark.parametrize("w,h,c,ch", SIZES)
def test_project(w, h, c, ch, odd_values):
    require_gpu()
    print(f"project {w}x{h} C {c}", flush=True)
    _, ring, den = _scene(w, h, c, ch, odd_values)
    cells = (w // 8) * (h // 8)
    want = np.full(9 * cells * 9, -7.0, np.float32)
    d_history, d_ring, d_den = dev(want), dev(ring), dev(den)
    words = dev(O.grain_pattern_words().view(np.int32))
    L.check(L.load().avd_site_grain_project(_p(d_ring), _p(d_den), _p(words), _p(d_history), w, h, c, ch, 1, 4, 1, None))
    with np.errstate(all="ignore"):
        O.grain_project(ring, den, w, h, c, ch, 1, want, 4)
    _same(host(d_history), want, "history")


@pytest.mark.parametrize("cells", [0, 1, 128, 129, 1023, 1024, 1025, 2176])
@pytest.mark.parametrize("at", [0, 1, 3])
def test_reduce(cells, at):
    require_gpu()
    print(f"reduce {cells} cells at float {at}", flush=True)
    rng = np.random.default_rng(cells)
    part = rng.standard_normal((cells, 48)).astype(np.float32)
    part[:, 47] = rng.choice([0, 1, 7, 15, 16, 99, -2, 4.7, np.nan], cells)
    chunk = rng.standard_normal(3 + 16 * 47).astype(np.float32)
    buf, d_chunk = dev(np.concatenate([np.zeros(at, np.float32), part.reshape(-1), np.ones(1, np.float32)])), dev(chunk)
    L.check(L.load().avd_site_grain_reduce(_p(buf[at:]), cells, _p(d_chunk), 3, None))
    want = O.grain_reduce(part.reshape(-1), chunk, 3) if cells else chunk
    _same(host(d_chunk), want, cells)

"""The f64 grain fit on the GPU against the oracle where its pivot rule and its guards decide: equal
pivots (the last row in the swapped order wins), rows swapped in every column, zero and negative zero
lags, NaN and infinite lags, more records than workgroups resident at once."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import avd

import oracle as O
from gpu_helpers import dev, host, require_gpu

pytestmark = pytest.mark.gpu


def _records(kind):
    rng = np.random.default_rng(len(kind))
    out = []
    for k in range(12):
        lags = np.zeros(46)
        if kind == "ties":  # no correction (zero lag 0): entries of equal magnitude everywhere
            lags[1:] = rng.choice([-1.0, 1.0], 45)
        elif kind == "few values":
            lags[1:] = rng.choice([-2.0, 0.0, 0.5, 2.0], 45)
        elif kind == "negative":
            lags[:] = rng.uniform(-1, 1, 46)
            lags[0] = -abs(lags[0])
        elif kind == "not finite":
            lags[:] = rng.uniform(-0.2, 0.2, 46)
            lags[0] = 1.0 if k % 3 else 0.0
            lags[1 + k * 3] = [np.nan, np.inf, -np.inf][k % 3]
        elif kind == "tiny":
            lags[:] = rng.uniform(-1, 1, 46) * 10.0 ** -(8 + k)
            lags[0] = 0.0
        out.append(np.r_[lags, 640.0 if k != 5 else -1.0])
    return np.array(out * (40 if kind == "ties" else 1))


@pytest.mark.parametrize("kind", ["ties", "few values", "negative", "not finite", "tiny"])
def test_fit_pivots_as_the_oracle(kind):
    require_gpu()
    print(f"grain fit, {kind}", flush=True)
    records = _records(kind)
    n = len(records)
    outs = [torch.zeros(n, 47, dtype=torch.float64, device="cuda"), torch.zeros(n, 24, dtype=torch.float64, device="cuda"),
            torch.zeros(n, 24, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda"),
            torch.zeros(n, dtype=torch.int32, device="cuda")]
    rec = dev(records)
    avd._lib.check(avd.load().avd_site_grain_fit(ctypes.c_void_p(rec.data_ptr()), n,
                                                 *[ctypes.c_void_p(t.data_ptr()) for t in outs], None))
    with np.errstate(all="ignore"):
        want = O.grain_fit(records)
    for got, exp in zip((host(t) for t in outs), want):
        exp = np.asarray(exp).astype(got.dtype).reshape(got.shape)
        assert np.array_equal(got, exp, equal_nan=got.dtype.kind == "f")

"""What the launch tuner's comparison of NLM window candidates can see: on the content it fills its buffers
with, a window that reads a wrong row, column, frame or confidence gives other weight sums almost everywhere
(the mistakes are made in the oracle's inputs)."""
from __future__ import annotations

import numpy as np
import pytest

import avd
import oracle as O


def _content(shape, confidence, first, P, h2, offset):
    lib = avd.load()
    n = int(np.prod(shape))
    return np.array([lib.avd_tuning_sample_for_test(confidence, first + i, P, h2, offset) for i in range(n)],
                    np.float32).reshape(shape)


@pytest.mark.parametrize("strength,offset", [(1.2, 0.0), (8.0, 0.01)])
@pytest.mark.parametrize("W,H,C,P,S", [(24, 20, 1, 0, 1), (21, 18, 2, 2, 2), (24, 20, 1, 4, 2), (20, 22, 2, 8, 1)])
def test_a_wrong_index_shows(W, H, C, P, S, strength, offset):
    h2 = float(O.h2_inv_norm(strength, P))
    centre, fwd, bwd = (_content((H, W, C), 0, k * W * H * C, P, h2, offset) for k in range(3))
    bx, by = -(-W // 8), -(-H // 8)
    conf = [_content((by, bx), 1, k * bx * by, P, h2, offset) for k in range(2)]
    lut = O.spatial_offset_lut(S, offset)

    def pair(c=centre, f=fwd, b=bwd, cf=conf[0], cb=conf[1]):
        out = [np.zeros(W * H * C), np.zeros(W * H), np.zeros(W * H)]
        O.nlm_pair(*(np.ascontiguousarray(x.reshape(-1)) for x in (c, f, b)), W, H, C, P, S, h2, offset,
                   np.ascontiguousarray(cf.reshape(-1)), np.ascontiguousarray(cb.reshape(-1)), 8, bx, by, *out,
                   precision="f64")
        return out[1]

    def single(c=centre):
        out = [np.zeros(W * H * C), np.zeros(W * H), np.zeros(W * H)]
        O.nlm_single(np.ascontiguousarray(c.reshape(-1)), W, H, C, P, S, h2, lut, *out, precision="f64")
        return out[1]

    def differ(a, b):
        return np.mean(np.abs(a - b) > 1e-5 * np.maximum(np.abs(a), 1e-3))

    right = pair()
    for axis in (0, 1):  # a row or a column off, of either frame and of the confidences
        assert differ(right, pair(f=np.roll(fwd, 1, axis))) > 0.9
        assert differ(right, pair(b=np.roll(bwd, 1, axis))) > 0.9
        assert differ(right, pair(cf=np.roll(conf[0], 1, axis))) > 0.9
        assert differ(right, pair(cb=np.roll(conf[1], 1, axis))) > 0.9
        assert differ(right, pair(c=np.roll(centre, 1, axis))) > 0.9
        assert differ(single(), single(c=np.roll(centre, 1, axis))) > 0.9
    assert differ(right, pair(f=bwd, b=fwd)) > 0.9
    assert differ(right, pair(cf=conf[1], cb=conf[0])) > 0.9
    if C == 2:
        assert differ(right, pair(f=fwd[..., ::-1])) > 0.9

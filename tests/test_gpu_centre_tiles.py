"""The matrix-core centre search against the oracle, word for word: frames whose rectangles clip on every
side, one column or row of positions, odd widths (both copies of the code plane), reference grids that do
not fill a wave's 2 x 4 block, search rectangles up to the two tiles' 31 columns, contents of exact
duplicates (the reference itself is not the first of them), and the largest products and sums the
accumulators meet (codes of 0 and 1023 alone)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from gpu_helpers import assert_members_equal, collab_pass, dev, require_gpu, site_collab_search

pytestmark = pytest.mark.gpu


def _codes(w, h, c, content):
    rng = np.random.default_rng(w * 31 + h + c)
    if content == "noise":
        return rng.integers(0, 1024, (h, w, c))
    if content == "extremes":
        return rng.integers(0, 2, (h, w, c)) * 1023
    if content == "black":
        return np.zeros((h, w, c))
    if content == "white":
        return np.full((h, w, c), 1023)
    if content == "edge":  # the best candidates of a reference share a column
        return 300 + 400 * (np.arange(w)[None, :, None] > w // 2) + rng.integers(0, 9, (h, w, c))
    x, y = np.arange(w)[None, :, None], np.arange(h)[:, None, None]
    return (x // 4 * 131 + y // 5 * 57 + 0 * np.arange(c)) % 1024  # "blocks"


@pytest.mark.parametrize("group", [8, 16])
@pytest.mark.parametrize("content", ["noise", "extremes", "black", "white", "edge", "blocks"])
@pytest.mark.parametrize("w,h,c,step,s", [(8, 8, 1, 4, 9), (8, 8, 2, 4, 9), (9, 8, 1, 1, 15), (8, 41, 1, 3, 12),
                                          (8, 40, 2, 3, 12), (43, 9, 2, 4, 12), (57, 45, 1, 4, 12), (56, 47, 2, 3, 14),
                                          (51, 39, 1, 3, 1), (61, 33, 1, 8, 11), (33, 34, 2, 8, 11)])
def test_members(w, h, c, step, s, content, group):
    require_gpu()
    print(f"centre {w}x{h} C {c} step {step} S {s} {content} {group}", flush=True)
    codes = np.ascontiguousarray(_codes(w, h, c, content), np.uint16).reshape(1, -1)
    geom = O.MotionGeom(w, h, 16, 8, 4, 2)
    p = collab_pass(w, h, c, 0, s, 2, 0.05, 2.7, 0.01, 2.0, 0, 1, geom, code_bits=10, step=step, group_size=group)
    op = O.collab_params(w, h, c, 0, s, 2, 0.05, 2.7, 0.01, 2.0, geom, step=step, group_size=group)
    want = O.collab_search(codes, op, 0, [], None, None)
    got = site_collab_search(p, codes=dev(codes.view(np.int16)))
    assert_members_equal(got, want, "members", group_size=group)

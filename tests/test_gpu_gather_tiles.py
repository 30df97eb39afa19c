"""The tile gather at the edges of its 32x32 tiles against the oracle, bit for bit: frames of whole tiles,
of one pixel more and of part tiles, one and two channels, eight and sixteen members, lists longer than
the 256 entries of a batch and far shorter ones."""
from __future__ import annotations

import numpy as np
import pytest

import avd
import oracle as O
from avd import _lib as L
from gpu_helpers import require_gpu, run_engine, words_dev
from test_gpu_k16 import _opts, _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,step", [(8, 4), (16, 3)])
@pytest.mark.parametrize("w,h", [(32, 32), (33, 39), (64, 40), (71, 65)])
def test_engine(w, h, group, step):
    require_gpu()
    print(f"gather {w}x{h} group {group}", flush=True)
    depth, r, s, frames, sigma = 10, 1, 6, 4, 16.0 / 1023
    clip = avd.synth.clip(frames, w, h, depth, 505 + w, chroma="444", sigma_luma=16.0, sigma_chroma=8.0)
    geom = L.Geometry(w, h, 3, L.SampleFormat.u16(10), L.SampleFormat.u16(10), 0)
    opts = _opts(r, s, sigma, step, group)
    eng = avd.build_engine("nl4d", geom, luma=opts, chroma=opts)
    got = run_engine(eng, [[words_dev(p.numpy(), depth) for p in f] for f in clip], depth, [(w, h)] * 3)
    pl = O.Nl4dPass(_spec(r, s, sigma, step, group), w, h, 1, depth, depth)
    pc = O.Nl4dPass(_spec(r, s, sigma, step, group), w, h, 2, depth, depth)
    O.link_motion(pl, pc, "444")
    want_l, _ = O.run_stream(pl, [[O.pack_plane(f[0].numpy(), depth)] for f in clip])
    want_c, _ = O.run_stream(pc, [[O.pack_plane(f[1].numpy(), depth), O.pack_plane(f[2].numpy(), depth)] for f in clip])
    for i in range(frames):
        for k, want in enumerate((want_l[i][0], want_c[i][0], want_c[i][1])):
            assert np.array_equal(got[i][k], want), (i, k)

"""A batch's trace takes four lanes per ray where its frames together have at most 384 x 384 pixels
(393 216 where they are path-traced), one lane otherwise, and the deepest octrees first: every
session's frame and visit count equals the plain path's, at the edges of both, for mixed depths and
both shadings in one submit."""
import numpy as np
import pytest

import temporalsetinversion_amd as T
from temporalsetinversion_amd import _lib, scenes
from temporalsetinversion_amd.batch import Batch

pytestmark = pytest.mark.gpu

CIN = _lib.TSI_SHADE_CINEMATIC
VIEW = T.look_at_inverse((2.2, 1.7, 2.6))
TIME = float(np.float32(0.2))


@pytest.mark.parametrize("frames", [   # (width, height, localsubdiv, tape, shading)
    [(1, 1, 4, 0, 0)],
    [(384, 384, 5, 1, 0)],
    [(383, 385, 5, 0, 0)],
    [(384, 384, 5, 1, 0), (1, 1, 6, 0, 0)],
    [(5, 3, 3, 0, 0), (64, 33, 6, 1, 0), (7, 9, 5, 0, 0), (4, 4, 1, 1, 0)],
    [(384, 385, 4, 0, 0), (20, 13, 5, 1, CIN), (33, 7, 4, 0, CIN), (9, 2, 6, 1, 0)],
    [(640, 616, 3, 1, CIN), (31, 17, 5, 0, 0)],
])
def test_batched_frames_equal_the_plain_ones(frames):
    tapes = [T.tape_from_ll(x) for x in scenes.batch_test_sets()["pair"]]
    with Batch(tapes, arena_bytes=len(frames) * (64 << 20) + (64 << 20), max_sessions=len(frames)) as b:
        sids = [b.open(tape=tape, localsubdiv=L, voxel_capacity=1 << 18, max_width=w, max_height=h, shading=shading)
                for w, h, L, tape, shading in frames]
        res, _, _ = b.run([(sid, TIME, f[0], f[1], VIEW) for sid, f in zip(sids, frames)])
        got = [b.frame(sid, f[0], f[1]) for sid, f in zip(sids, frames)]
    for (w, h, L, tape, shading), r, (rgba, depth) in zip(frames, res, got):
        print(f"{w}x{h} L{L} tape {tape} shading {shading}", flush=True)
        with T.State(tapes[tape], width=w, height=h, localsubdiv=L, shading=shading, prune=False,
                     voxel_capacity=1 << 18) as st:
            st.reset()
            st.update(TIME, VIEW)
            st.set_inversion()
            want, wdepth = st.trace()
            assert r["status"] == 0 and r["node_visits"] == st.last_trace()[1]
        assert np.array_equal(rgba.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(depth.view(np.uint32), wdepth.view(np.uint32))

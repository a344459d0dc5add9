"""Frames of more rows than a launch's grid holds (65 535 tiles of 4 pixels with four lanes per ray, of 8 with
one) are traced by the persistent form: the same pixels as a batch's, whose blocks are numbered in one dimension."""
import numpy as np
import pytest

import temporalsetinversion_amd as T
from temporalsetinversion_amd import _lib, scenes
from temporalsetinversion_amd.batch import Batch

pytestmark = pytest.mark.gpu

VIEW = T.look_at_inverse((2.2, 1.7, 2.6))
TIME = float(np.float32(0.2))


@pytest.mark.parametrize("height,shading", [(262140, _lib.TSI_SHADE_CINEMATIC), (262141, _lib.TSI_SHADE_CINEMATIC),
                                            (524280, 0), (524281, 0)])
@pytest.mark.parametrize("overlap", [False, True])
def test_frames_of_one_column(height, shading, overlap):
    tape = T.tape_from_ll(scenes.batch_test_sets()["one"][0])
    with Batch([tape], arena_bytes=128 << 20, max_sessions=1) as b:
        sid = b.open(tape=0, localsubdiv=5, voxel_capacity=1 << 18, max_width=1, max_height=height, shading=shading)
        (r,), _, _ = b.run([(sid, TIME, 1, height, VIEW)])
        want = b.frame(sid, 1, height)
    assert (want[1] > 0).sum() > 1000
    with T.State(tape, width=1, height=height, localsubdiv=5, shading=shading, prune=False, voxel_capacity=1 << 18) as st:
        st.reset()
        st.update(TIME, VIEW)
        st.set_inversion()
        if overlap:
            st.render_async()
            got = st.trace_wait()
        else:
            got = st.trace()
        assert st.last_trace()[1] == r["node_visits"]
    for x, y in zip(got, want):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))

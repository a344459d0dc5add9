"""An allocation that fails is reported once, by the call that made it, and not by the next one."""
import numpy as np
import pytest

import oracle
import temporalsetinversion_amd as T
from helpers import assert_same_nodes, tape_of
from temporalsetinversion_amd import scenes
from temporalsetinversion_amd.batch import Batch

pytestmark = pytest.mark.gpu


def _batch():
    Batch([T.tape_from_ll(x) for x in scenes.batch_test_sets()["one"]], arena_bytes=1 << 42, max_sessions=1)


def _frame():
    with T.State(tape_of("spheres"), width=1, height=1, localsubdiv=4, voxel_capacity=1 << 16) as st:
        st.uniforms.resolution[0] = st.uniforms.resolution[1] = 1 << 20   # 18 TB
        st.reset()
        st.update(0.0)
        st.trace(pixels=False)


@pytest.mark.parametrize("allocate", [_batch, _frame])
def test_the_next_call_works(allocate):
    tape = tape_of("spheres")
    fr = oracle.Frame(tape, localsubdiv=5, voxel_capacity=1 << 18)
    with T.State(tape, width=32, height=24, localsubdiv=5, voxel_capacity=1 << 18) as st:
        st.reset()
        for k, t in enumerate([0.0, 0.25]):
            with pytest.raises(T.TsiError) as e:
                allocate()
            assert e.value.code == -1                      # TSI_E_OOM
            st.update(float(np.float32(t)))
            st.set_inversion()
            fr.set_inversion(t)
            assert_same_nodes(st.read_nodes(), fr.export(), f"frame {k}")
            st.enqueue_root()
            fr.enqueue_root()
    fr.close()

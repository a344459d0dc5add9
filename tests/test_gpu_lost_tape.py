"""A context whose tape's kernels or buffers are gone (a rebuild that failed, an upload without the memory for it)
refuses frames until a tape is uploaded, and computes the oracle's frames after that."""
import numpy as np
import pytest

import oracle
import temporalsetinversion_amd as T
from helpers import assert_same_nodes, tape_of
from temporalsetinversion_amd import scenes
from test_chain_domain import shells
from test_gpu_memory_limits import _HoldAllBut

pytestmark = pytest.mark.gpu

JIT, NO_TAPE, OOM = -11, -8, -1


def _upload(st, tape):
    buf = (T._lib.GpuInstruction * len(tape)).from_buffer_copy(np.ascontiguousarray(tape).tobytes())
    T.check(T.lib().tsi_upload_tape(st._ctx, buf, len(tape)), "tsi_upload_tape")
    st.tape = tape


def _fails(code, call):
    with pytest.raises(T.TsiError) as e:
        call()
    assert e.value.code == code


def _matches_the_oracle(st, tape, L):
    fr = oracle.Frame(tape, localsubdiv=L, voxel_capacity=1 << 20)
    st.reset()
    for k, t in enumerate([0.0, 1 / 60]):
        st.update(float(np.float32(t)))
        st.set_inversion()
        fr.set_inversion(float(np.float32(t)))
        assert_same_nodes(st.read_nodes(), fr.export(), f"frame {k}")
        st.enqueue_root()
        fr.enqueue_root()
    fr.close()


@pytest.mark.parametrize("which", ["straight", "chain"])
def test_kernels_that_cannot_be_rebuilt(which, monkeypatch, tmp_path):
    """A frame past t = 64 needs other kernels (a chain's: where it is none any more, past t = 4096); the compiler
    is given an option that it does not know."""
    monkeypatch.setenv("TSI_JIT_CACHE", str(tmp_path))
    tape = tape_of("sphere") if which == "straight" else shells(19, link="min")
    with T.State(tape, width=16, height=16, localsubdiv=5, voxel_capacity=1 << 18) as st:
        _matches_the_oracle(st, tape, 5)
        monkeypatch.setenv("HIPRTC_COMPILE_OPTIONS_APPEND", "-fno-such-option")
        try:
            st.update(71.5 if which == "straight" else 5000.0)
            _fails(JIT, st.set_inversion)
        finally:
            monkeypatch.setenv("HIPRTC_COMPILE_OPTIONS_APPEND", "")
        for t in (71.5, 0.0):
            st.update(t)
            _fails(NO_TAPE, st.set_inversion)
            _fails(NO_TAPE, lambda: T.check(T.lib().tsi_set_inversion_async(st._ctx), "tsi_set_inversion_async"))
        st.trace(pixels=False)                      # the octree is still there
        assert len(st.read_nodes()) > 1
        _upload(st, tape)
        _matches_the_oracle(st, tape, 5)


@pytest.mark.parametrize("engine", ["interpreter", "compiled"])
def test_upload_without_the_memory(engine):
    """csg's saved-operand stack takes 10 GB; 4 are free."""
    small, large = tape_of("spheres"), T.tape_from_ll(scenes.SCENES["csg"]())
    with T.State(small, width=16, height=16, localsubdiv=5, voxel_capacity=1 << 18, engine=engine, prune=False) as st:
        _matches_the_oracle(st, small, 5)
        with _HoldAllBut(4 << 30):
            _fails(OOM, lambda: _upload(st, large))
            st.update(0.1)
            _fails(NO_TAPE, st.set_inversion)
            _upload(st, small)                      # fits
            _matches_the_oracle(st, small, 5)
        _upload(st, large)
        st.reset()
        st.update(0.1)
        assert st.set_inversion().stats["cell_evals"] > 0

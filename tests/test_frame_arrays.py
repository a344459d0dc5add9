"""Frames in pooled pinned host memory (tsi_host_buffer): what a frame's arrays hold does not depend on
where they lie (pinned, pageable and staged, pageable and direct), a buffer in use is never handed out
again, an array larger than the frame is 0 beyond it, and the pool's bound holds."""
import ctypes as C
import threading

import numpy as np
import pytest

import temporalsetinversion_amd as T
from helpers import tape_of


def test_no_buffers_without_a_context():
    assert not T.lib().tsi_host_buffer(1 << 20)
    T.lib().tsi_host_buffer_free(None)
    a = T._lib.frame_array((3, 5), np.float32, 0)
    assert a.shape == (3, 5) and not a.any() and a.flags.writeable


def _frame(st, w, h):
    st.uniforms.resolution[0], st.uniforms.resolution[1] = w, h
    st.width, st.height = w, h
    st.update(0.0)
    return st.trace()


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(1, 1), (37, 21), (160, 160), (300, 301), (1024, 512)])   # staged up to 512 KiB
def test_frames_are_the_same_wherever_they_are_copied(w, h):
    with T.State(tape_of("spheres"), width=w, height=h, localsubdiv=6, voxel_capacity=1 << 18) as st:
        st.reset()
        st.update(0.0)
        st.set_inversion()
        rgba, depth = _frame(st, w, h)
        again = st.trace_wait()
        a, b = np.full((h, w, 4), 7, np.float32), np.full((h, w), 7, np.float32)
        T.check(T.lib().tsi_trace_wait(st._ctx, a.ctypes.data, b.ctypes.data), "tsi_trace_wait")
        for x, y in ((rgba, a), (depth, b), (again[0], a), (again[1], b)):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
        # half pinned, half pageable; one of the two alone
        c = np.full((h, w), 7, np.float32)
        T.check(T.lib().tsi_trace_wait(st._ctx, None, c.ctypes.data), "tsi_trace_wait")
        assert np.array_equal(b, c)
        T.check(T.lib().tsi_trace_wait(st._ctx, again[0].ctypes.data, c.ctypes.data), "tsi_trace_wait")
        assert np.array_equal(again[0].view(np.uint32), a.view(np.uint32))
        img, ref = st.frame_rgba8(), np.full((h, w, 4), 7, np.uint8)
        T.check(T.lib().tsi_frame_rgba8(st._ctx, ref.ctypes.data), "tsi_frame_rgba8")
        assert np.array_equal(img, ref)
        # arrays larger than the frame
        st.height = h + 3
        rgba2, depth2 = st.trace_wait()
        st.height = h
        assert np.array_equal(rgba2[:h].view(np.uint32), a.view(np.uint32)) and not rgba2[h:].any() and not depth2[h:].any()


@pytest.mark.gpu
def test_buffers_are_bounded_and_outlive_their_context():
    lib = T.lib()
    with T.State(tape_of("spheres"), width=64, height=48, localsubdiv=5, voxel_capacity=1 << 18) as st:
        st.reset()
        st.update(0.0)
        st.set_inversion()
        kept = [st.trace()[0] for _ in range(4)]
        assert len({x.ctypes.data for x in kept}) == 4            # all in use
        sizes, held = [384 << 20, 384 << 20, 384 << 20], []
        for s in sizes:                                           # 1 GiB in all, kept's included
            p = lib.tsi_host_buffer(s)
            held.append(p)
        assert held[0] and held[1] and not held[2]
        assert lib.tsi_host_buffer((1 << 30) + 1) is None
        for p in held[:2]:
            C.memset(p, 1, 384 << 20)
            lib.tsi_host_buffer_free(p)
        # several threads
        seen, lock = [], threading.Lock()

        def take():
            for k in range(50):
                p = lib.tsi_host_buffer(65536 * (1 + k % 3))
                with lock:
                    assert p not in seen
                    seen.append(p)
                C.memset(p, 3, 65536)
                with lock:
                    seen.remove(p)
                lib.tsi_host_buffer_free(p)
        threads = [threading.Thread(target=take) for _ in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    first = kept[0].copy()
    assert all(np.array_equal(x, first) for x in kept)            # the context is gone, the frames are not
    kept.clear()
    assert not lib.tsi_host_buffer(65536)

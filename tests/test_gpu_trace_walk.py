"""The trace's fast walk (tsi_trace.hip): its division core against the compiler's correctly rounded
division, and frames of rays that it cannot take or takes at the edge (zero direction components,
steps along several axes at once, a camera inside the box, an empty octree, a deep one), in both ray
layouts (frames up to 32 768 pixels use four lanes per ray), bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle
import temporalsetinversion_amd as T
from helpers import run_pair, tape_of

pytestmark = pytest.mark.gpu


def _check_div(first, count, recip):
    fn = T.lib().tsi_check_div
    fn.restype = C.c_int
    fn.argtypes = [C.c_uint32, C.c_uint32, C.c_int32, C.POINTER(C.c_uint64), C.POINTER(C.c_uint32), C.POINTER(C.c_uint32)]
    bad, first_bad, done = C.c_uint64(0), C.c_uint32(0), C.c_uint32(0)
    T.check(fn(first, count, recip, C.byref(bad), C.byref(first_bad), C.byref(done)), "tsi_check_div")
    print(f"first {first:#x} recip {recip}: {done.value} compared, {bad.value} differ (first {first_bad.value:#x})", flush=True)
    assert done.value == count
    return bad.value


def test_reciprocal_of_every_moderate_float():
    lo = int(np.float32(2.0 ** -30).view(np.uint32))
    hi = int(np.float32(2.0 ** 30).view(np.uint32))
    assert _check_div(lo, hi - lo + 1, 1) == 0
    assert _check_div(lo | 0x80000000, hi - lo + 1, 1) == 0


@pytest.mark.parametrize("stream", [1, 2])
def test_division_of_moderate_floats(stream):
    assert _check_div(stream, 1 << 30, 0) == 0


# (view, frame): straight down -z (rays with zero components on odd sizes, ties on the diagonals and
# between symmetric sides), the (1, 1, 1) diagonal (x == z on the middle column), inside the box
VIEWS = [((0.0, 0.0, 6.0), (41, 41)), ((0.0, 0.0, 6.0), (64, 64)), ((4.0, 4.0, 4.0), (33, 24)),
         ((0.05, 0.02, 0.9), (40, 31)), ((0.0, 0.0, 6.0), (201, 171)), ((4.0, 4.0, 4.0), (225, 160))]


@pytest.mark.parametrize("eye,size", VIEWS)
@pytest.mark.parametrize("scene,L", [("sphere", 5), ("spheres", 6)])
def test_frames_of_degenerate_rays_match_the_oracle(eye, size, scene, L):
    view = T.look_at_inverse(eye)
    W, H = size
    for k, g, o, gs, os_, gf, of in run_pair(tape_of(scene), [0.0, 0.25], width=W, height=H, trace_every=1,
                                                localsubdiv=L, view=view):
        for a, b, what in ((gf[0], of[0], "colour"), (gf[1], of[1], "depth")):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"{what} differs in frame {k}"


def test_deep_octree_matches_the_oracle():
    """More levels than the ray's stack has entries (the reference drops pushes on a full stack):
    a thin sub-box keeps the octree small."""
    tape = oracle.parse_ll(_tiny_sphere())
    view = T.look_at_inverse((0.02, 0.015, 0.03))
    for k, g, o, gs, os_, gf, of in run_pair(tape, [0.0], width=24, height=16, trace_every=1, localsubdiv=17, view=view):
        assert o["depth"].max() == 17
        for a, b, what in ((gf[0], of[0], "colour"), (gf[1], of[1], "depth")):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"{what} differs in frame {k}"


def _tiny_sphere():
    from temporalsetinversion_amd import scenes
    return scenes.sphere_unit(0.0005)


def test_empty_octree():
    with T.State(tape_of("sphere"), width=20, height=12, localsubdiv=4, voxel_capacity=1 << 16) as st:
        st.reset()
        st.update(0.0, T.look_at_inverse((0.0, 0.0, 12.0)))
        rgba, depth = st.trace()
        assert np.all(depth == -1.0) and np.all(rgba == 1.0)

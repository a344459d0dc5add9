"""The trace's routes by frame size: four lanes per ray up to kQuadPixels (kQuadPixelsCinematic where
frames are path-traced), one lane per ray above, as a full launch where the call waits for it and as 12
persistent wavefronts per CU over a snapshot where it overlaps the next set inversion; $TSI_TRACE_BLOCKS
forces the persistent form, which is always one lane per ray.  Sizes are derived from the thresholds in the
source.

* rays that the fast walk cannot take or takes at the edge (zero direction components, steps along several
  axes at once, a camera inside the box, an octree deeper than the ray's stack): one lane per ray, both
  forms, bit for bit against the oracle (test_gpu_trace_walk.py has them with four lanes);
* overlapped traces, two frames in flight: the frames and visits of traces that are waited for."""
import os
import re

import numpy as np
import pytest

import oracle
import temporalsetinversion_amd as T
from helpers import run_pair, tape_of
from temporalsetinversion_amd import _lib, scenes

pytestmark = pytest.mark.gpu

CIN = _lib.TSI_SHADE_CINEMATIC
GRADIENTS = _lib.TSI_SHADE_NORMALS | _lib.TSI_SHADE_GRADIENT


def _thresholds():
    src = open(os.path.join(_lib.HERE, "csrc", "tsi_trace.hip")).read()
    m = re.search(r"kQuadPixels = (\d+), kQuadPixelsCinematic = (\d+);", src)
    return int(m.group(1)), int(m.group(2))


QUAD, QUAD_CINEMATIC = _thresholds()


def _above(pixels, odd):
    """The smallest square of an odd or even side above `pixels`."""
    side = int(np.sqrt(pixels)) + 1
    side += side % 2 != odd
    assert side * side > pixels
    return side, side


@pytest.fixture(params=["persistent", "full"])
def form(request, monkeypatch):
    """One lane per ray: (name, smallest frame)."""
    if request.param == "persistent":
        monkeypatch.setenv("TSI_TRACE_BLOCKS", "1")   # read when a context is created
    else:
        monkeypatch.delenv("TSI_TRACE_BLOCKS", raising=False)
    return request.param


def _compare(tape, times, size, view, L):
    hits = 0
    for k, g, o, gs, os_, gf, of in run_pair(tape, times, width=size[0], height=size[1], trace_every=1, localsubdiv=L,
                                             view=view):
        for a, b, what in ((gf[0], of[0], "colour"), (gf[1], of[1], "depth")):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"{what} differs in frame {k}"
        hits += int((of[1] > 0).sum())
    assert hits > 0


# straight down -z (odd sizes: zero components; even: ties on the diagonals), the (1, 1, 1) diagonal
# (x == z on the middle column), inside the box
VIEWS = [((0.0, 0.0, 6.0), (41, 41)), ((0.0, 0.0, 6.0), (64, 64)), ((4.0, 4.0, 4.0), (33, 24)),
         ((4.0, 4.0, 4.0), (64, 48)), ((0.05, 0.02, 0.9), (40, 31))]


@pytest.mark.parametrize("eye,size", VIEWS)
@pytest.mark.parametrize("scene,L", [("sphere", 5), ("spheres", 6)])
def test_degenerate_rays_with_one_lane_per_ray(form, eye, size, scene, L):
    if form == "full":
        size = _above(QUAD, size[0] % 2)
    _compare(tape_of(scene), [0.0, 0.25], size, T.look_at_inverse(eye), L)


# (so close that rays end on the surface: 1 of 24x16 and about 700 of 386x386)
DEEP_VIEW = T.look_at_inverse((0.002, 0.0015, 0.003))


def test_deep_octree_with_one_lane_per_ray(form):
    size = _above(QUAD, 0) if form == "full" else (24, 16)
    _compare(oracle.parse_ll(scenes.sphere_unit(0.0005)), [0.0], size, DEEP_VIEW, 17)


@pytest.mark.parametrize("size", [(24, 16), (64, 64)])
def test_deep_octree_with_four_lanes_per_ray(monkeypatch, size):
    monkeypatch.delenv("TSI_TRACE_BLOCKS", raising=False)
    _compare(oracle.parse_ll(scenes.sphere_unit(0.0005)), [0.0], size, DEEP_VIEW, 17)


@pytest.mark.parametrize("shading,pixels", [(0, QUAD), (GRADIENTS, QUAD), (CIN, QUAD_CINEMATIC)])
@pytest.mark.parametrize("above", [False, True])
def test_overlapped_traces_equal_blocking_ones(monkeypatch, shading, pixels, above):
    monkeypatch.delenv("TSI_TRACE_BLOCKS", raising=False)
    w, h = _above(pixels, 1)
    if not above:
        h = pixels // w
    assert (w * h > pixels) == above
    tape = T.tape_from_ll(scenes.SCENES["spheres"]())
    view = T.look_at_inverse((2.2, 1.7, 2.6))
    times = [float(np.float32(0.1 + k / 30.0)) for k in range(3 if shading == CIN else 5)]
    kw = dict(width=w, height=h, localsubdiv=6, shading=shading, voxel_capacity=1 << 18)
    want, visits = [], []
    with T.State(tape, **kw) as st:
        st.reset()
        for t in times:
            st.update(t, view)
            st.set_inversion()
            want.append(st.render())
            visits.append(st.last_trace()[1])
    assert not np.array_equal(want[0][1], want[-1][1])
    for n in range(2, len(times) + 1):
        with T.State(tape, **kw) as st:
            st.reset()
            for k, t in enumerate(times[:n]):
                st.update(t, view)
                st.set_inversion_async()
                st.render_async()
                if k > 0:
                    st.set_inversion_result()
            st.set_inversion_result()
            got = st.trace_wait()
            _, total, count = st.trace_totals()
        assert (total, count) == (sum(visits[:n]), n)
        for a, b in zip(got, want[n - 1]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))

"""Chains where values meet fix's clamp at +-1e6.  It clamps an interval's two bounds apart, so one beyond
comes out reversed, and a decision of a cell's parents need not hold in the cell: a tape is a chain only on a
domain where no value is clamped, and kernels leave the chain when a frame leaves the domain."""
import ctypes as C

import numpy as np
import pytest

import temporalsetinversion_amd as T
from helpers import assert_same_nodes
from temporalsetinversion_amd import scenes
from test_chain import frames, is_chain


def shells(n, scale=1.0, warp=None, motion=0.1, link="smin"):
    """n thin spheres in coordinates scaled or warped, joined by smooth minima (or minima)."""
    rng = np.random.default_rng(n)
    B = scenes.Tape()
    x, y, z = B.x, B.y, B.mul(B.z, scale)
    if warp:
        z = B.add(z, warp(B))
    d = None
    for i in range(n):
        c = rng.uniform(-0.9, 0.9, 3)
        q = [B.sub(B.sub(x, float(c[0])), B.mul(B.t, motion * float(c[1]))), B.sub(y, float(c[1])), B.sub(z, float(c[2]))]
        prim = B.sub(B.length3(*q), float(rng.uniform(0.1, 0.4)))
        d = prim if d is None else (B.smin(d, prim, 0.3) if link == "smin" else B.min(d, prim))
    return T.tape_from_ll(B.to_ll(d))


def log_warp(B):   # -inf and NaN around a cylinder
    return B.mul(B._call1("logf", B.sub(B.sq(B.x), 0.15)), 0.02)


CLAMPED = {"scaled": shells(20, 1000.0), "log": shells(18, 1.0, log_warp), "fast": shells(20, motion=60.0)}


def test_tapes_that_may_clamp_are_no_chains():
    assert is_chain(shells(20)) and is_chain(shells(20, 100.0)) and is_chain(shells(20, link="min"))
    assert is_chain(shells(20, motion=10.0))                         # 640 at t = 64
    # the root of a negative number is 0, not NaN
    B = scenes.Tape()
    d = B.sub(B.x, 3.0)
    for i in range(20):
        d = B.min(d, B.sub(B.sqrt(B.sub(B.add(B.sq(B.sub(B.x, 0.1 * i)), B.sq(B.z)), 0.01)), 0.1))
    assert is_chain(T.tape_from_ll(B.to_ll(d)))
    for name, tape in CLAMPED.items():
        assert not is_chain(tape), name


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CLAMPED))
def test_tapes_that_clamp_match_the_full_tape(name):
    times = [0.0, 1 / 60, 0.1, 0.05] if name != "fast" else [1.0, 17.0, 17.0 + 1 / 60, 40.0]
    kw = dict(localsubdiv=6, lipschitz_corrected=True)
    ref = frames(CLAMPED[name], times, engine="interpreter", prune=False, **kw)
    got = frames(CLAMPED[name], times, prune=False, **kw)
    for k, ((gs, g), (rs, r)) in enumerate(zip(got, ref)):
        assert_same_nodes(g, r, f"{name} frame {k}")
        assert gs["cell_evals"] == rs["cell_evals"]
    assert sum(len(r) for _, r in ref) > 100


def _frames(tape, times, boxes=None, **kw):
    out = []
    with T.State(tape, voxel_capacity=1 << 20, localsubdiv=6, **kw) as st:
        for k, t in enumerate(times):
            if k == 0 or (boxes and boxes[k] != boxes[k - 1]):
                T.check(T.lib().tsi_reset(st._ctx, (C.c_float * 6)(*(boxes[k] if boxes else (-5, -5, -5, 5, 5, 5)))), "reset")
            st.update(float(np.float32(t)))
            out.append((st.set_inversion().stats, st.read_nodes(), st.tape_info()))
            st.enqueue_root()
    return out


def _compare(tape, times, boxes=None, **kw):
    ref = _frames(tape, times, boxes, engine="interpreter", prune=False, **kw)
    got = _frames(tape, times, boxes, prune=True, **kw)
    for k, ((gs, g, _), (rs, r, _)) in enumerate(zip(got, ref)):
        print(f"frame {k}: t {times[k]}, {len(r)} nodes, {gs['pruned_instr']} records left out", flush=True)
        assert_same_nodes(g, r, f"frame {k}")
        for key in ("cell_evals", "rev_evals", "rev_ops", "parents", "enqueued", "deallocs", "allocated_nodes"):
            assert gs[key] == rs[key], f"frame {k}: {key}"
    return got


@pytest.mark.gpu
@pytest.mark.parametrize("swept", [False, True])
def test_animations_that_leave_the_domain(swept):
    """Past t = 64 the kernels are rebuilt for a wider domain, as a chain while no value can be clamped there
    (0.9 t squared: 8.5e5 at 1 024, beyond 1e6 at 16 384), else without one."""
    tape = shells(20, motion=1.0, link="min")
    assert is_chain(tape)
    times = [0.0, 1 / 60, 63.99, 64.01, 64.03, 255.0, 256.5, 300.0, 5000.0, 5000.02, 0.5]
    got = _compare(tape, times, swept_volume=swept, swept_window=0.1)
    assert [i["specialized"] for _, _, i in got] == [1] * 8 + [0] * 3
    first = [s for s, _, _ in got]
    assert first[0]["pruned_instr"] > 0 and first[8]["pruned_instr"] == 0


@pytest.mark.gpu
def test_root_boxes_that_leave_the_domain():
    """A box beyond +-5 (still a chain), one beyond any, and one turned over on an axis."""
    tape = shells(20, link="min")
    boxes = [(-5, -5, -5, 5, 5, 5), (-7, -1, -1, 1, 1, 1), (-1, -1, -1, 1, 1, 1), (1, -1, -1, -1, 1, 1), (-3e3, -1, -1, 3e3, 1, 1)]
    got = _compare(tape, [0.0, 0.1, 0.2, 0.25, 0.3], boxes)
    assert [i["specialized"] for _, _, i in got] == [1, 1, 1, 0, 0]


@pytest.mark.gpu
def test_batched_windows_that_leave_the_domain():
    """A swept window reaches from the frame's time to swept_window before it; one of negative length, after it."""
    from temporalsetinversion_amd.batch import Batch
    tapes = [T.tape_from_ll(x) for x in scenes.batch_test_sets()["one"]]
    with Batch(tapes, arena_bytes=64 << 20, max_sessions=2) as b:
        kw = dict(tape=0, localsubdiv=4, voxel_capacity=1 << 16, max_width=16, max_height=16, swept_volume=True)
        before, after = b.open(swept_window=10.0, **kw), b.open(swept_window=-10.0, **kw)
        for sid, t, inside in ((before, 64.0, True), (before, 64.1, False), (before, 7.9, False), (before, 8.0, True),
                               (after, 54.0, True), (after, 54.1, False), (after, -2.0, True), (after, -2.1, False),
                               (before, float("nan"), False)):
            if inside:
                (r,), _, _ = b.run([(sid, t, 0, 0, None)])
                assert r["status"] == 0
            else:
                with pytest.raises(T.TsiError) as e:
                    b.run([(sid, t, 0, 0, None)])
                assert e.value.code == -6                 # TSI_E_ARG

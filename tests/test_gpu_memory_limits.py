"""Records of chain tapes only save work: where device memory is nearly spent they give way to what a batch's
or a context's calls need, and the results are the same without them."""
import ctypes as C
import time

import numpy as np
import pytest

import temporalsetinversion_amd as T
from temporalsetinversion_amd import scenes
from temporalsetinversion_amd.batch import Batch

pytestmark = pytest.mark.gpu

MIB = 1 << 20
VIEW = T.look_at_inverse((2.2, 1.7, 2.6))


def _free_now():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert T.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # (of the runtime that the library is bound to)
    return free.value


def _free():
    """Free device memory, once it has not changed for a second (the driver clears what is given back first)."""
    seen = [_free_now()]
    while (len(seen) < 6 or len(set(seen[-6:])) > 1) and len(seen) < 100:
        time.sleep(0.2)
        seen.append(_free_now())
    return seen[-1]


class _HoldAllBut:
    """Allocations that leave at most `rest` bytes and 8 MiB free."""

    def __init__(self, rest):
        self.held = []
        for _ in range(20):
            extra = _free() - rest
            if extra <= 8 * MIB:
                break
            p = C.c_void_p()
            assert T.lib().hipMalloc(C.byref(p), C.c_size_t(extra - 4 * MIB)) == 0
            self.held.append(p)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.held:
            T.lib().hipFree(p)


def _state(**kw):
    return T.State(T.tape_from_ll(scenes.SCENES["csg"]()), width=16, height=16, localsubdiv=7, prune=False,
                   voxel_capacity=1 << 22, queue_capacity=ENTRIES, **kw)


ENTRIES = 12_500_000   # 3.2 GB of records
WIDTH = 16384


def _frames(st, overlap, height):
    """Nodes and counts of two frames, the second after (or beside) the first's trace of WIDTH x height pixels."""
    out = []
    st.reset()
    for k, size in enumerate([(WIDTH, height), (16, 16)]):
        st.uniforms.resolution[0], st.uniforms.resolution[1] = size
        st.update(0.25 + k / 60.0, VIEW)
        s = st.set_inversion().stats
        out.append([s[k] for k in ("cell_evals", "rev_evals", "parents", "enqueued", "allocated_nodes")])
        if overlap:
            st.render_async()
        else:
            st.render(pixels=False)
    st.trace_wait(pixels=False)
    nodes = st.read_nodes()
    order = np.lexsort((nodes["k"], nodes["j"], nodes["i"], nodes["depth"]))
    return out, nodes[order].tobytes()


@pytest.fixture(scope="module")
def sizes():
    """Bytes of the records, and of a context without them (what a process keeps beside it not counted)."""
    with _state(prune_capacity=ENTRIES) as st:
        _frames(st, True, 64)
        with_records = _free()
    with _state(prune_capacity=8) as st:
        _frames(st, True, 64)
        without = _free()
    return without - with_records, _free() - without


@pytest.mark.parametrize("overlap", [False, True])
def test_frame_that_needs_the_records_memory(sizes, overlap):
    """The records fit their share of what is free, and the frame's pixels (25 GB) do not fit beside them.
    Whichever of them is there, half the records' size stays free for what a launch needs."""
    records, base = sizes
    assert records > 3 << 30
    room = 8 * records + (2 << 30)     # free beside a context without records
    height = (room - records // 2) // (20 * WIDTH)
    print(f"{records >> 20} MiB of records, {room >> 20} free, a frame of {WIDTH}x{height}", flush=True)
    with _state() as st:
        want = _frames(st, overlap, height)
    with _HoldAllBut(base + room):
        with _state(prune_capacity=ENTRIES) as st:
            got = _frames(st, overlap, height)
    assert got == want


def _batch_frame(b, tape):
    sid = b.open(tape=tape, localsubdiv=7, voxel_capacity=1 << 19, max_width=64, max_height=48)
    stats = []
    for t in (0.25, 0.27):
        (s,), _, _ = b.run([(sid, t, 64, 48, VIEW, t == 0.25)])
        assert s["status"] == 0
        stats.append([s[k] for k in ("cell_evals", "rev_evals", "parents", "enqueued", "allocated_nodes", "node_visits")])
    return (stats, *b.frame(sid, 64, 48))


def test_batch_arena_that_leaves_two_gibibytes():
    """The records of 1024 sessions of these tapes would take 3.9 GB."""
    tapes = [T.tape_from_ll(t) for t in scenes.served_tapes()]
    longest = int(np.argmax([len(t) for t in tapes]))
    before = _free()
    with Batch(tapes, arena_bytes=256 * MIB, max_sessions=2) as b:
        used = before - _free()   # its records are a few MB
        want = _batch_frame(b, longest)
    arena = _free() - used - 2048 * MIB
    print(f"arena of {arena >> 20} MiB, {_free() >> 20} free", flush=True)
    with Batch(tapes, arena_bytes=arena, max_sessions=1024) as b:
        got = _batch_frame(b, longest)
    assert got[0] == want[0]
    assert all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(got[1:], want[1:]))

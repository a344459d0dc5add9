"""Performance cases of the framework: what its users have it do, through its public interface.

Three kinds of pass:

* "clip": an animation on one context (`State`): the octree is reset, then `frames` frames at
  t0 + k/60, each a set inversion, the trace of the frame and the root's re-enqueue.  `loop` is how
  the program drives it: "sync" waits for every frame (`compute` + `render`, the reference's frame
  loop), "async" keeps two frames in flight (`set_inversion_async` / `render_async`).  `out` is what
  it takes of a frame: "pixels" (colour and depth copied to the host, `render`'s default), "rgba8"
  (the frame dump's bytes) or "device" (the frame stays on the GPU).
* "requests": independent requests on a `Batch`, each a session started from an empty octree, all in
  one submit, then every session's frame copied out (`Batch.frame`, the only way to a session's
  pixels).
* "served": the sessions of a `Batch` over `frames` consecutive submits of their next 1/60 window,
  the way the server's loop runs them, then every session's last frame copied out.

The seed gives the camera (a direction around the scene, at the case's distance), the start time of
the animation and the requests' times; tapes, depths, frame sizes and options are the case's.  Tapes
are those that the build compiles ahead, so that no pass or preparation holds a compilation.  Every
case also returns the frames' work counts (whole numbers).  The outputs follow from decisions on
binary32 intervals (which cells the octree splits); no 64-bit computation gives the same octree, so
`exact` has no value for them: they are held to the start's, bit for bit in practice.
"""
from __future__ import annotations

import ctypes

import numpy as np
import torch

import temporalsetinversion_amd as T
from temporalsetinversion_amd import scenes
from temporalsetinversion_amd.batch import Batch

COUNTS = ("cell_evals", "rev_evals", "parents", "deallocs", "enqueued", "allocated_nodes")

# tapes the build compiles ahead (text, surface area of the field's zero set in box units: what
# the number of cells follows from)
TAPES = {
    "sphere": (lambda: scenes.sphere_unit(1.0), 12.6),
    "spheres": (lambda: scenes.SCENES["spheres"](), 2.6),
    "spheres_linear": (lambda: scenes.SCENES["spheres_linear"](), 2.6),
    "capsules": (lambda: scenes.SCENES["capsules"](), 7.0),
    "csg": (lambda: scenes.SCENES["csg"](), 14.0),
    "mixed6": (lambda: scenes.mixed(11, 6), 8.0),
    "mixed10": (lambda: scenes.mixed(12, 10), 8.0),
    "mixed14": (lambda: scenes.mixed(13, 14), 8.0),
    "mixed20": (lambda: scenes.mixed(14, 20), 8.0),
}
# tape sets whose batch module the build compiles ahead
SETS = {
    "one": lambda: scenes.batch_test_sets()["one"],
    "pair": lambda: scenes.batch_test_sets()["pair"],
    "mixed4": lambda: scenes.batch_test_sets()["mixed4"],
    "batched": scenes.batch_tapes,
    "served": scenes.served_tapes,
}
# pool of a session by its depth (twice that of the deepest request met at the depth)
CAPACITY = {4: 1 << 16, 5: 1 << 17, 6: 1 << 19, 7: 1 << 20, 8: 1 << 21, 9: 1 << 22}


def clip(name, scene, L, w, h, frames, *, swept=False, lipschitz=False, shading=0, prune=True, engine="compiled",
         loop="sync", out="device", dist=12.0, capacity=1 << 24):
    return dict(name=name, kind="clip", scene=scene, L=L, w=w, h=h, frames=frames, swept=swept, lipschitz=lipschitz,
                shading=shading, prune=prune, engine=engine, loop=loop, out=out, dist=dist, capacity=capacity)


def batch(name, kind, tapes, count, L0, L1, w, h, frames, mix, dist=12.0):
    return dict(name=name, kind=kind, tapes=tapes, count=count, L0=L0, L1=L1, w=w, h=h, frames=frames, mix=mix, dist=dist)


def listed():
    return [
        # the smallest call: a still object, one frame from an empty octree (a thumbnail)
        clip("thumbnail", "sphere", 4, 64, 48, 1, out="pixels", dist=4.0, capacity=1 << 18),
        # a small interactive preview: the reference's CPU configuration, every frame waited for and
        # its pixels taken
        clip("preview", "spheres", 6, 256, 256, 8, out="pixels", capacity=1 << 20),
        # the plain method at 512^3: 64 capsules, Lipschitz correction, two frames in flight
        clip("capsules_512", "capsules", 9, 1024, 1024, 12, lipschitz=True, prune=False, loop="async"),
        # the plain method at 1024^3: 256-primitive CSG, swept windows, full HD, two frames in flight
        clip("csg_1024", "csg", 10, 1920, 1080, 8, swept=True, prune=False, loop="async"),
        # the frame dump loop with a context's default options (every frame to RGBA8), odd size, near
        clip("dump_capsules", "capsules", 8, 801, 599, 8, out="rgba8", dist=4.0),
        # default options on a long tape
        clip("default_csg", "csg", 8, 1280, 720, 6),
        # surface normals from the reverse pass: every cell is differentiated; a tape with divisions
        clip("normals_mixed", "mixed20", 8, 1024, 768, 4, shading=3, loop="async", dist=5.0),
        # a scene evaluated without compiling its tape (an editor's loop)
        clip("interpreted", "spheres_linear", 7, 640, 480, 6, swept=True, engine="interpreter"),
        # the path tracer, gradient normals off
        clip("cinematic", "csg", 8, 641, 361, 2, swept=True, shading=4, prune=False, out="pixels", dist=5.0),
        # independent requests over 16 tapes, mixed depths and frame sizes, one submit
        batch("requests_24", "requests", "batched", 24, 6, 9, 640, 480, 1, 6),
        # a full server: 32 scenes' next windows, submit after submit
        batch("served_28", "served", "served", 28, 7, 9, 512, 512, 6, 12),
        # a server with one client: one session's frames, each waited for
        batch("served_1", "served", "pair", 1, 7, 7, 320, 240, 8, 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["clip", "clip", "clip", "requests", "served"])
    dist = round(rng.uniform(4.0, 12.0), 2)
    if kind == "clip":
        scene = rng.choice(sorted(TAPES))
        engine = rng.choice(["compiled", "compiled", "compiled", "interpreter"])
        prune = rng.random() < 0.5
        shading = rng.choice([0, 0, 0, 0, 1, 3, 4])
        # long tapes, the interpreter and default pruning keep to the depths they are used at
        top = {"csg": 9, "sphere": 9}.get(scene, 9) - (1 if prune and scene == "csg" else 0)
        top -= 2 if engine == "interpreter" else 0
        top -= 1 if shading == 4 else 0
        L = rng.randint(4, top)
        w, h = _log_int(rng, 48, 1280), _log_int(rng, 40, 800)
        if shading == 4:
            w, h = max(48, w // 2), max(40, h // 2)
        case = clip("", scene, L, w, h, _log_int(rng, 1, 8), swept=rng.random() < 0.4, lipschitz=rng.random() < 0.4,
                    shading=shading, prune=prune, engine=engine, loop=rng.choice(["sync", "async"]),
                    out=rng.choice(["device", "pixels", "rgba8"]), dist=dist, capacity=1 << (20 if L <= 6 else 24))
    else:
        tapes = rng.choice(["pair", "mixed4", "batched"] if kind == "requests" else ["one", "pair", "served"])
        L0 = rng.randint(4, 8)
        case = batch("", kind, tapes, _log_int(rng, 1, 24), L0, min(9, L0 + rng.randint(0, 2)), _log_int(rng, 64, 720),
                     _log_int(rng, 64, 512), 1 if kind == "requests" else _log_int(rng, 1, 6), rng.randint(0, 1 << 20), dist)
    del case["name"]
    return case


def _camera(rng, dist):
    a, z = rng.uniform(0.0, 2.0 * np.pi), rng.uniform(-0.7, 0.7)
    r = np.sqrt(1.0 - z * z)
    return T.look_at_inverse((dist * r * np.cos(a), dist * z, dist * r * np.sin(a)))


def _time(t):
    return float(np.float32(t))


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    view = _camera(rng, case["dist"])
    t0 = rng.uniform(0.0, 1.0)
    if case["kind"] == "clip":
        st = T.State(TAPES[case["scene"]][0](), width=case["w"], height=case["h"], localsubdiv=case["L"],
                     swept_volume=case["swept"], lipschitz_corrected=case["lipschitz"], prune=case["prune"],
                     engine=case["engine"], shading=case["shading"], voxel_capacity=case["capacity"])
        times = [_time(t0 + k / 60.0) for k in range(case["frames"])]
        return dict(case=case, st=st, view=view, times=times)
    tapes = [T.tape_from_ll(x) for x in SETS[case["tapes"]]()]
    mix = np.random.default_rng(case["mix"])   # the case's mix of requests: tapes, depths, sizes
    b = None
    sessions, room = [], 0
    for i in range(case["count"]):
        L = int(mix.integers(case["L0"], case["L1"] + 1))
        s = float(mix.uniform(0.6, 1.0))
        w, h = max(16, int(case["w"] * s)), max(16, int(case["h"] * s))
        kw = dict(tape=int(mix.integers(0, len(tapes))), localsubdiv=L, voxel_capacity=CAPACITY[L], max_width=w,
                  max_height=h)
        if case["kind"] == "requests":
            window = _time(mix.uniform(1.0 / 30.0, 0.5))
            kw.update(swept_volume=True, swept_window=window)
            t = [_time(rng.uniform(window, 1.0))]
        else:
            kw.update(lipschitz_corrected=True)
            t = [_time(t0 + k / 60.0) for k in range(case["frames"])]
        sessions.append((kw, w, h, t))
        room += 100 * CAPACITY[L] + 24 * w * h + (8 << 20)
    b = Batch(tapes, arena_bytes=room, max_sessions=case["count"])
    b.tune(waves_per_simd=b.info()["max_waves_per_simd"])
    sids = [b.open(**kw) for kw, _, _, _ in sessions]
    submits = [[(sid, t[k], w, h, view, k == 0) for sid, (_, w, h, t) in zip(sids, sessions)]
               for k in range(case["frames"])]
    return dict(case=case, b=b, submits=submits)


class _DeviceArray:
    """Device memory of the library, for torch (the array interface).  Torch keeps this object as long
    as a tensor of it, and this object the context whose memory it is."""

    def __init__(self, st, ptr, shape):
        self.owner = st
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=3)


def _device_frame(st):
    rgba, depth = ctypes.c_void_p(), ctypes.c_void_p()
    T.check(T.lib().tsi_frame_device(st._ctx, ctypes.byref(rgba), ctypes.byref(depth)), "tsi_frame_device")
    return (torch.as_tensor(_DeviceArray(st, rgba.value, (st.height, st.width, 4)), device="cuda"),
            torch.as_tensor(_DeviceArray(st, depth.value, (st.height, st.width)), device="cuda"))


def _counts(stats):
    return np.array([[s[k] for k in COUNTS] for s in stats], np.int64)


def _run_clip(state):
    case, st, view = state["case"], state["st"], state["view"]
    stats, frame = [], None
    st.reset()
    if case["loop"] == "sync":
        for t in state["times"]:
            st.update(t, view)
            stats.append(st.set_inversion().stats)
            frame = st.render(pixels=case["out"] == "pixels")
            if case["out"] == "rgba8":
                frame = st.frame_rgba8()
        visits = [st.last_trace()[1]]
    else:
        inflight = 0
        for t in state["times"]:
            st.update(t, view)
            st.set_inversion_async()
            st.render_async()
            inflight += 1
            if inflight == 2:
                stats.append(st.set_inversion_result().stats)
                inflight -= 1
        while inflight:
            stats.append(st.set_inversion_result().stats)
            inflight -= 1
        frame = st.trace_wait(pixels=case["out"] == "pixels")
        if case["out"] == "rgba8":
            frame = st.frame_rgba8()
        visits = [st.last_trace()[1]]
    if case["out"] == "device":
        frame = _device_frame(st)
    return dict(frame=frame, counts=_counts(stats), visits=np.array(visits, np.int64))


def run(state):
    if state["case"]["kind"] == "clip":
        return _run_clip(state)
    b, stats = state["b"], []
    for frames in state["submits"]:
        res, _, _ = b.run(frames)
        stats += res
    for s in stats:
        if s["status"] != 0:
            raise T.TsiError(s["status"], "a session's frame")
    images = [b.frame(sid, w, h) for sid, _, w, h, _, _ in state["submits"][-1]]
    return dict(frames=images, counts=_counts(stats), visits=np.array([s["node_visits"] for s in stats], np.int64))


def exact(case, seed):
    return None


def _cells(area, L, frames, swept):
    """Cells of a clip: a leaf level's cells that the surface crosses (its area over a leaf's face,
    times 1.5 for its slant), 8 children for each crossed parent of every level above; later
    frames touch about 0.4 of that."""
    leaves = 1.5 * area * (2.0 ** L / 10.0) ** 2
    full = 8.0 / 3.0 * leaves + 8.0 * L
    return full * (1.0 + 0.4 * (frames - 1)) * (1.2 if swept else 1.0)


def work(case):
    """Operations: each cell evaluates the tape (a record of an interval is about 4 operations, and
    about as many again to differentiate half of the cells).  Bytes: a cell's 64-byte state written
    once, each frame's pixels written once (20 B) with about 20 node reads of 16 B for each."""
    if case["kind"] == "clip":
        text, area = TAPES[case["scene"]]
        jobs = [(text().count("\n"), area, case["L"], case["w"] * case["h"], case["frames"])]
        swept, rays = case["swept"], 16 if case["shading"] & 4 else 1
    else:
        n = np.mean([x.count("\n") for x in SETS[case["tapes"]]()])
        s = 0.65   # the mean of the sizes' squared scale
        jobs = [(n, 4.0, (case["L0"] + case["L1"]) / 2.0, s * case["w"] * case["h"], case["frames"])] * case["count"]
        swept, rays = case["kind"] == "requests", 1
    flops = nbytes = 0.0
    for records, area, L, pixels, frames in jobs:
        cells = _cells(area, L, frames, swept)
        flops += cells * records * 6.0 + pixels * frames * rays * 500.0
        nbytes += cells * 64.0 + pixels * frames * (20.0 + rays * 320.0)
    return {"bytes": nbytes, "flops": flops}

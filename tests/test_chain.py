"""Unions compiled as chains: loops over segments that leave out the segments a cell's parents have
decided.  Which tapes are taken (CPU, from the generated source), and that nodes and statistics are
those of the interpreter running the full tape, bit for bit, over the forms a chain accepts: links by
min, max and smooth min with the chain on either side, 17 to 140 segments (a mask word holds 32),
several structures of segments, literals shared and not, moving by t alone (linear, sine) and through
sines of the position, and with every option that changes a cell's inputs or t-window."""
import numpy as np
import pytest

import temporalsetinversion_amd as T
from helpers import assert_same_nodes
from temporalsetinversion_amd import scenes


def union(n, links, motion="linear", seed=0, head=None, shared=False):
    """n primitives (spheres, boxes, slabs) joined by the links in turn: 'min', 'max' (a carved
    primitive), 'smin', 'rmin' / 'rsmin' (the chain is the right operand)."""
    rng = np.random.default_rng(seed)
    B = scenes.Tape()
    x, y, z = B.x, B.y, B.z
    if motion == "warp":
        x = B.add(B.x, B.mul(B.sin(B.add(B.mul(B.y, 2.0), B.t)), 0.05))
        z = B.add(B.z, B.mul(B.cos(B.mul(B.x, 3.0)), 0.05))
    d = None
    for i in range(n):
        c = rng.uniform(-0.9, 0.9, 3)
        q = []
        for a, p in enumerate((x, y, z)):
            if motion == "static" or (motion == "warp" and a == 1):
                q.append(B.sub(p, float(c[a])))
            elif motion == "sine":
                q.append(B.sub(p, B.add(B.mul(B.sin(B.add(B.t, float(c[a]))), 0.1), float(c[a]))))
            else:
                q.append(B.sub(B.sub(p, float(c[a])), B.mul(B.t, float(rng.uniform(-0.3, 0.3)))))
        kind, r = i % 3, float(rng.uniform(0.03, 0.15))
        if kind == 0:
            prim = B.sub(B.length3(*q), r)
        elif kind == 1:
            prim = B.max(B.max(B.sub(B.abs(q[0]), r), B.sub(B.abs(q[1]), 0.06)), B.sub(B.abs(q[2]), r))
        else:
            prim = B.sub(B.sqrt(B.add(B.sq(q[0]), B.sq(q[2]))), r) if shared else B.sub(B.abs(q[1]), 0.3 * r)
            prim = B.max(prim, B.sub(B.length3(*q), 2 * r))
        if d is None:
            d = prim
            continue
        link = links[i % len(links)]
        if link == "min":
            d = B.min(d, prim)
        elif link == "rmin":
            d = B.min(prim, d)
        elif link == "smin":
            d = B.smin(d, prim, 0.05)
        elif link == "rsmin":
            d = B.smin(prim, d, float(rng.uniform(0.02, 0.06)))
        else:
            d = B.max(d, B.neg(prim))
    if head:
        d = head(B, d)
    return T.tape_from_ll(B.to_ll(d))


def is_chain(tape):
    return "kSkip = true" in T.kernel_source(tape, prune=False)[0]


def test_which_tapes_are_chains():
    assert is_chain(union(20, ["min"]))
    assert is_chain(union(20, ["smin", "max", "rmin", "rsmin"]))
    assert is_chain(union(20, ["min"], "sine")) and is_chain(union(20, ["smin"], "warp"))
    assert not is_chain(union(8, ["min"]))                       # few segments: a straight line
    # the output is not the union itself (its sign is, but not its bits)
    assert not is_chain(union(20, ["min"], head=lambda B, d: B.mul(d, 0.5)))
    # a position's sine inside a segment: decisions are not inherited to the ulp
    B = scenes.Tape()
    d = B.sub(B.length3(B.x, B.y, B.z), 0.1)
    for i in range(20):
        d = B.min(d, B.sub(B.length2(B.sub(B.x, 0.1 * i), B.sin(B.mul(B.y, 1.0 + i))), 0.1))
    assert not is_chain(T.tape_from_ll(B.to_ll(d)))
    # own operands that read the chain's operand
    B = scenes.Tape()
    d = B.sub(B.length3(B.x, B.y, B.z), 0.1)
    for i in range(20):
        d = B.min(d, B.mul(B.add(d, 0.1 + i), B.x))
    assert not is_chain(T.tape_from_ll(B.to_ll(d)))
    # a value made inside one segment and read by another
    B = scenes.Tape()
    d = B.sub(B.length3(B.x, B.y, B.z), 0.1)
    for i in range(20):
        q = B.sub(B.x, 0.05 * i)
        d = B.min(d, B.sub(B.length2(q, B.y), 0.1))
        d = B.min(d, B.sub(B.length2(q, B.z), 0.1))
    assert not is_chain(T.tape_from_ll(B.to_ll(d)))
    # the bound of the sensitivities' growth along smooth minima: 2 c h = 1/2 each, 2^100 at most
    for n, chain in ((160, True), (180, False)):
        B = scenes.Tape()
        d = B.sub(B.length2(B.x, B.y), 0.1)
        for i in range(n):
            d = B.smin(d, B.sub(B.length2(B.sub(B.x, 0.01 * (i + 1)), B.z), 0.1), 0.05)
        assert is_chain(T.tape_from_ll(B.to_ll(d))) == chain


def frames(tape, times, **kw):
    out = []
    with T.State(tape, voxel_capacity=1 << 20, **kw) as st:
        st.reset()
        for k, t in enumerate(times):
            st.update(float(np.float32(t)))
            out.append((st.set_inversion().stats, st.read_nodes()))
            st.enqueue_root()
    return out


# forward in equal and unequal steps, the same time twice, backwards, past what the octree knows
TIMES = [0.0, 1 / 60, 2 / 60, 2 / 60, 0.1, 0.11, 0.05, 0.6, 0.62]

CASES = {
    "min20": (union(20, ["min"]), {}),
    "min32-static": (union(32, ["rmin", "min"], "static", 1), {}),
    "mix33": (union(33, ["smin", "max", "rmin", "rsmin", "min"], seed=2), {}),
    "mix64-swept": (union(64, ["min", "smin"], seed=3), dict(swept_volume=True, swept_window=0.03)),
    "mix65-sine": (union(65, ["smin", "rmin", "max"], "sine", 4), {}),
    "sine-swept": (union(24, ["rsmin", "min"], "sine", 5), dict(swept_volume=True, swept_window=0.05)),
    "warp": (union(40, ["min", "smin", "max"], "warp", 6), {}),
    "warp-lipschitz": (union(40, ["rmin"], "warp", 7), dict(lipschitz_corrected=True, fast_multiplier=0.3)),
    "gradients": (union(48, ["smin"], seed=8), dict(shading=3)),
    "no-fast": (union(36, ["min", "rsmin"], seed=9), dict(fastenabled=False, point_sample=False)),
    "small-records": (union(36, ["min", "max"], seed=10), dict(prune_capacity=64)),
    "no-speculation": (union(36, ["smin", "min"], seed=11), dict(speculate=False)),
    "mix140": (union(140, ["min", "smin", "rmin", "max"], seed=12, shared=True), dict(localsubdiv=6)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_chains_match_the_full_tape(case):
    tape, kw = CASES[case]
    assert is_chain(tape)
    kw = {"localsubdiv": 7, **kw}
    ref = frames(tape, TIMES, engine="interpreter", prune=False, **{k: v for k, v in kw.items() if k != "prune_capacity"})
    for prune in (False, True):
        got = frames(tape, TIMES, prune=prune, **kw)
        for k, ((gs, g), (rs, r)) in enumerate(zip(got, ref)):
            print(f"{case} prune={prune} frame {k}: {len(r)} nodes, {gs['fwd_ops']} of {rs['fwd_ops']} ops", flush=True)
            assert_same_nodes(g, r, f"{case} prune={prune} frame {k}")
            for key in ("cell_evals", "rev_evals", "rev_ops", "parents", "enqueued", "deallocs", "allocated_nodes"):
                assert gs[key] == rs[key], f"frame {k}: {key}"
            if not prune:   # pruning refused: the whole tape's counts
                assert gs["fwd_ops"] == rs["fwd_ops"] and gs["pruned_instr"] == 0
            elif k == 0:    # new cells' parents have decided most segments
                assert gs["fwd_ops"] < rs["fwd_ops"] and gs["pruned_instr"] > 0


@pytest.mark.gpu
def test_batched_chains_match_the_plain_path():
    """Chains of several record lengths, and tapes that are none, in one batch: sessions of different
    tapes run side by side (each wavefront's columns have the room of the longest record)."""
    from temporalsetinversion_amd.batch import Batch
    tapes = [union(20, ["min"]), union(120, ["smin", "min"], "linear", 3), union(65, ["smin", "rmin"], "sine", 4),
             union(40, ["min", "max"], "warp", 6), union(6, ["min"], "static", 9)]
    sessions = [(0, 6, {}), (1, 6, dict(lipschitz_corrected=True)), (2, 6, {}), (3, 6, {}), (4, 5, {}),
                (1, 5, dict(swept_volume=True, swept_window=0.2)), (2, 6, dict(swept_volume=True, swept_window=0.1)),
                (3, 5, dict(point_sample=False)), (1, 7, {})]
    times = [0.0, 1 / 60, 2 / 60, 0.2, 0.15]
    with Batch(tapes, arena_bytes=sum(100 << 18 for _ in sessions) + (256 << 20), max_sessions=len(sessions)) as b:
        sids = [b.open(tape=t, localsubdiv=L, voxel_capacity=1 << 18, max_width=16, max_height=16, **kw)
                for t, L, kw in sessions]
        got = []
        for k, t in enumerate(times):
            res, _, _ = b.run([(sid, float(np.float32(t + 0.01 * i)), 0, 0, None) for i, sid in enumerate(sids)])
            got.append([(r, b.read_nodes(sid)) for r, sid in zip(res, sids)])
    for i, (t, L, kw) in enumerate(sessions):
        want = frames(tapes[t], [x + 0.01 * i for x in times], localsubdiv=L, engine="interpreter", prune=False, **kw)
        for k, (rs, r) in enumerate(want):
            gs, g = got[k][i]
            assert gs["status"] == 0
            assert_same_nodes(g, r, f"session {i} frame {k}")
            for key in ("cell_evals", "rev_evals", "fwd_ops", "rev_ops", "parents", "enqueued", "deallocs", "allocated_nodes"):
                assert gs[key] == rs[key], f"session {i} frame {k}: {key}"

"""tsi_stats.eval_kernel_ms by the device's clock: from a level's first block to its last, on frontiers
of more blocks than the chip holds."""
import pytest

import temporalsetinversion_amd as T
from temporalsetinversion_amd import scenes

pytestmark = pytest.mark.gpu

SCENES = {"mixed20": lambda: scenes.mixed(14, 20), "csg": lambda: scenes.SCENES["csg"]()}


@pytest.mark.parametrize("scene,L,swept", [("mixed20", 10, False), ("csg", 10, True)])
def test_levels_are_timed_whole(scene, L, swept):
    """What the levels' span (events) holds beside them is a gap per level, shorter than a shallow level's whole
    launch (18 us at most).  (Not in a context's first frame, where the device waits for the host's first
    launches of each kernel.)"""
    with T.State(T.tape_from_ll(SCENES[scene]()), width=16, height=16, localsubdiv=L, swept_volume=swept, prune=False,
                 speculate=False, voxel_capacity=1 << 24) as st:
        for k in range(4):
            st.reset()
            st.update(0.25)
            s = st.set_inversion().stats
            print(f"{scene}: {s['cell_evals']} cells, levels {s['eval_kernel_ms']:.3f} of {s['eval_ms']:.3f} ms", flush=True)
            if k == 0:
                continue
            assert s["eval_ms"] > 0.3
            assert s["eval_ms"] - 0.018 * L <= s["eval_kernel_ms"] <= s["eval_ms"]

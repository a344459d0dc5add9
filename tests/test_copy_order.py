"""Copies out of the library wait for the work queued on their stream, wherever they go: into a pooled
array, through a staging buffer, or straight to pageable memory (tsi_frame_rgba8 queues its
conversion right before its copy)."""
import ctypes as C

import numpy as np
import pytest

import hostmem_stub
import temporalsetinversion_amd as T
from helpers import tape_of
from test_outputs import read_png

MAIN = r"""
int main(int argc, char **argv) {
    const size_t bytes = size_t(std::atoll(argv[1]));
    const bool pinned = std::strcmp(argv[2], "pinned") == 0, spent = argv[3][0] == 's';
    HostPoolUser user;
    // every byte of the pool handed out: no staging buffer
    std::vector<void *> held;
    if (spent)
        while (void *p = tsi_host_buffer(size_t(64) << 20)) held.push_back(p);
    Stream s;
    std::vector<char> src(bytes, 1), dst(bytes, 7), dst2(bytes, 7);
    char *to = pinned ? static_cast<char *>(tsi_host_buffer(bytes)) : dst.data();
    if (!to) return 2;
    s.queue.push_back([&] { std::memset(src.data(), 2, bytes); });   // the kernel before the copy
    const CopyOut out[2] = {{to, src.data(), bytes}, {dst2.data(), src.data(), bytes}};
    if (copy_out(out, 1, &s) != TSI_OK) return 3;
    for (size_t i = 0; i < bytes; ++i)
        if (to[i] != 2) { std::printf("byte %zu is %d\n", i, to[i]); return 4; }
    s.queue.push_back([&] { std::memset(src.data(), 3, bytes); });
    if (copy_out(out, 2, &s) != TSI_OK) return 5;
    for (size_t i = 0; i < bytes; ++i)
        if (to[i] != 3 || dst2[i] != 3) { std::printf("byte %zu is %d, %d\n", i, to[i], dst2[i]); return 6; }
    return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    return hostmem_stub.build(tmp_path_factory.mktemp("copies"), MAIN)


# up to 512 KiB in all is staged, beyond it and without a buffer copied directly
@pytest.mark.parametrize("bytes_", [1, 262144, 262145, 524288, 524289, 3 << 20])
@pytest.mark.parametrize("to,pool", [("pinned", "free"), ("pageable", "free"), ("pageable", "spent")])
def test_copies_come_after_the_stream(driver, bytes_, to, pool):
    hostmem_stub.run(driver, str(bytes_), to, pool)


def _rgba8(rgba):
    """The frame dump's conversion (k_rgba8): clamp to [0, 1], times 255 in binary32, half up."""
    x = np.minimum(np.maximum(rgba, np.float32(0.0)), np.float32(1.0)) * np.float32(255.0)
    return np.floor(x.astype(np.float64) + 0.5).astype(np.uint8)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(301, 200), (801, 599)])   # staged; 1.9 MB: directly
def test_rgba8_dumps_to_pageable_memory(tmp_path, w, h):
    """The first dump of a context, and one after the frame has changed, go to pageable memory."""
    for png in (False, True):
        with T.State(tape_of("spheres"), width=w, height=h, localsubdiv=6, voxel_capacity=1 << 18) as st:
            st.reset()
            last = None
            for k, eye in enumerate([(4.0, 3.0, 5.0), (-5.0, 2.0, 2.0), (0.5, 6.0, 1.0)]):
                st.update(0.25 * k, T.look_at_inverse(eye))
                st.set_inversion()
                st.render(pixels=False)
                if png:
                    path = tmp_path / f"{k}.png"
                    T.check(T.lib().tsi_save_frame_png(st._ctx, str(path).encode()), "tsi_save_frame_png")
                    out = read_png(path)
                else:
                    out = np.full((h, w, 4), 7, np.uint8)
                    T.check(T.lib().tsi_frame_rgba8(st._ctx, out.ctypes.data_as(C.c_void_p)), "tsi_frame_rgba8")
                assert np.array_equal(out, _rgba8(st.trace_wait()[0]))
                assert last is None or not np.array_equal(out, last)
                last = out

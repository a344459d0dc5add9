"""A forked process reads the frames its parent held (pinned memory is not inherited: the pool hands the
child copies at the same addresses), gives them back, and gets no pinned memory of its own."""
import os

import numpy as np
import pytest

import hostmem_stub
import temporalsetinversion_amd as T
from helpers import tape_of

MAIN = r"""
#include <pthread.h>
#include <sys/wait.h>
#include <unistd.h>
#include <atomic>
#include <thread>
static bool all(const char *p, size_t n, char v) {
    for (size_t i = 0; i < n; ++i)
        if (p[i] != v) return false;
    return true;
}
static int child(std::vector<std::pair<char *, size_t>> &held) {
    alarm(20);
    for (size_t k = 0; k < held.size(); ++k)
        if (!all(held[k].first, held[k].second, char(k + 1))) return 2;
    if (tsi_host_buffer(65536)) return 3;
    std::memset(held[0].first, 99, held[0].second);
    const pid_t pid = fork();   // and its own children
    if (pid == 0) _exit(all(held[0].first, held[0].second, 99) && all(held[1].first, held[1].second, 2) ? 0 : 1);
    int st = 0;
    waitpid(pid, &st, 0);
    if (st != 0) return 4;
    for (auto &h : held) tsi_host_buffer_free(h.first);
    return 0;
}
int main(int argc, char **argv) {
    const int threads = std::atoi(argv[1]);
    {
        HostPoolUser user;
        std::vector<std::pair<char *, size_t>> held;
        for (size_t n : {size_t(1), size_t(65536), size_t(65537), size_t(5) << 20, size_t(300000)}) {
            held.emplace_back(static_cast<char *>(tsi_host_buffer(n)), n);
            std::memset(held.back().first, int(held.size()), n);
        }
        tsi_host_buffer_free(tsi_host_buffer(1 << 20));   // one idle
        std::atomic<bool> stop{false};
        std::vector<std::thread> others;   // that may hold the pool's lock when the process forks
        for (int t = 0; t < threads; ++t)
            others.emplace_back([&] {
                while (!stop) tsi_host_buffer_free(tsi_host_buffer(70000));
            });
        int bad = 0;
        for (int k = 0; k < (threads ? 100 : 2) && !bad; ++k) {
            const pid_t pid = fork();
            if (pid == 0) _exit(child(held));
            waitpid(pid, &bad, 0);
        }
        stop = true;
        for (auto &t : others) t.join();
        if (bad) { std::printf("child: status %d\n", bad); return 2; }
        for (size_t k = 0; k < held.size(); ++k) {
            if (!all(held[k].first, held[k].second, char(k + 1))) return 3;
            tsi_host_buffer_free(held[k].first);
        }
    }
    return pinned_bytes() == 0 ? 0 : 4;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    return hostmem_stub.build(tmp_path_factory.mktemp("forked"), MAIN)


@pytest.mark.parametrize("threads", [0, 3])
def test_buffers_in_a_forked_process(driver, threads):
    hostmem_stub.run(driver, str(threads))


@pytest.mark.gpu
def test_frames_in_a_forked_process():
    frames = []
    with T.State(tape_of("spheres"), width=33, height=20, localsubdiv=6, voxel_capacity=1 << 18) as st:
        st.reset()
        st.update(0.0)
        st.set_inversion()
        for w, h in ((33, 20), (300, 301), (1280, 720)):
            st.uniforms.resolution[0], st.uniforms.resolution[1] = w, h
            st.width, st.height = w, h
            st.update(0.0)
            frames += [*st.trace(), st.frame_rgba8()]
        want = [f.copy() for f in frames]
        pid = os.fork()
        if pid == 0:   # reads, writes and drops them, without the GPU
            code = 1
            try:
                same = all(np.array_equal(f.view(np.uint8), x.view(np.uint8)) for f, x in zip(frames, want))
                frames[0][:] = 5.0
                frames.clear()
                code = 0 if same else 2
            finally:
                os._exit(code)
        assert os.waitpid(pid, 0)[1] == 0
        for f, x in zip(frames, want):
            assert np.array_equal(f.view(np.uint8), x.view(np.uint8))
        again = st.trace()
        assert np.array_equal(again[0].view(np.uint32), want[-3].view(np.uint32))

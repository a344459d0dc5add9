"""Running out of host memory anywhere in the pool of frame arrays: no exception leaves the library's C
entries, copies still arrive, and nothing stays pinned."""
import pytest

import hostmem_stub

MAIN = r"""
int main(int argc, char **argv) {
    const int first = std::atoi(argv[1]);
    std::vector<char> src(100000, 2), dst(100000);
    {
        HostPoolUser user;
        Stream s;
        s.queue.reserve(16);
        const CopyOut out{dst.data(), src.data(), src.size()};
        // what is pinned and idle, so that a buffer is reused (0), pinned (1), or pinned after others were
        // unpinned (2): the staging buffer of a copy
        const int how = std::atoi(argv[2]);
        std::vector<void *> held;
        held.reserve(64);
        if (how == 0) tsi_host_buffer_free(tsi_host_buffer(src.size()));
        if (how == 2) {
            for (int k = 0; k < 16; ++k) held.push_back(tsi_host_buffer(size_t(64) << 20));
            for (int k = 0; k < 4; ++k) { tsi_host_buffer_free(held.back()); held.pop_back(); }
        }
        allocations() = first;
        const int rc = copy_out(&out, 1, &s);
        allocations() = first;
        void *p = tsi_host_buffer(how == 2 ? size_t(200) << 20 : 70000);
        tsi_host_buffer_free(p);
        allocations() = -1;
        if (rc != TSI_OK || dst != src) return 3;
        for (void *x : held) tsi_host_buffer_free(x);
    }
    if (pinned_bytes() != 0) { std::printf("%zu bytes stay pinned\n", pinned_bytes()); return 4; }
    return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    return hostmem_stub.build(tmp_path_factory.mktemp("memory"), MAIN)


@pytest.mark.parametrize("how", [0, 1, 2])
@pytest.mark.parametrize("first", range(6))   # (no path allocates more than 4 times)
def test_no_memory_for_the_pool(driver, first, how):
    hostmem_stub.run(driver, str(first), str(how))

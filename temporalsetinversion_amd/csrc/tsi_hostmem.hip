// tsi_hostmem.hip -- see tsi_hostmem.h.
//
// A frame's pixels copied to pageable memory take a copy through the runtime's own staging: 110 us
// before the first byte (3.4 MB: 204 us, 262 KB: 113 us), and the page faults of a fresh array on
// top.  To pinned memory the same copies run at the link's rate: 68 us and 14 us.  So the arrays
// that the Python layer hands out are pinned buffers from a pool, and small copies to memory of the
// caller's go through a pinned buffer (262 KB: 14 us and a memcpy).  Pinning afresh for each frame
// costs 77 us for 4 MB and unpinning may wait for the device, hence a pool: bounded, shared by all
// threads, given back when the last context goes.  The bound is 25 full HD frames with their depth: a
// program that still held two submits' frames (95 MB each) while it took a third ran out of 256 MiB, and
// the third's copies took 13 ms instead of 2.7.
//
// A forked process does not inherit pinned memory (the driver's mapping is left out of the child), so a
// child that read its parent's frames would fault.  A fork therefore copies the buffers handed out
// (their contents once, into ordinary pages), and the child finds the copies at the same addresses; it
// gives them back as ordinary memory and gets no pinned memory of its own.
#include "tsi_hostmem.h"

#include <pthread.h>
#include <sys/mman.h>

#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <vector>

#include "tsi.h"

namespace tsi {
namespace {

constexpr size_t kPoolBytes = size_t(1) << 30;   // handed out and idle together
constexpr size_t kGrain = size_t(64) << 10;
constexpr size_t kStageBytes = size_t(512) << 10;  // pageable copies up to here are staged

struct Pool {
    std::mutex m;
    std::multimap<size_t, void *> idle;   // by size
    std::map<void *, size_t> out;
    size_t bytes = 0;
    int users = 0;
    char *stash = nullptr;                // during a fork: what the buffers handed out hold, one after the other
    size_t stash_bytes = 0;
    bool forked = false;                  // in a forked process: `out` is ordinary memory, `idle` is not mapped
};
Pool &pool();

// ---- forks (m is held from before the fork until after it, so that the child can use it) ----
void before_fork() {
    Pool &P = pool();
    P.m.lock();
    if (P.forked) return;
    for (const auto &x : P.out) P.stash_bytes += x.second;
    if (P.stash_bytes == 0) return;
    void *s = mmap(nullptr, P.stash_bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (s == MAP_FAILED) {   // (the child then has no frames)
        P.stash_bytes = 0;
        return;
    }
    P.stash = static_cast<char *>(s);
    size_t at = 0;
    for (const auto &x : P.out) {
        std::memcpy(P.stash + at, x.first, x.second);
        at += x.second;
    }
}

void after_fork_parent() {
    Pool &P = pool();
    if (P.stash) munmap(P.stash, P.stash_bytes);
    P.stash = nullptr;
    P.stash_bytes = 0;
    P.m.unlock();
}

void after_fork_child() {
    Pool &P = pool();
    P.forked = true;
    size_t at = 0;
    if (P.stash)
        for (const auto &x : P.out) {   // pages move, nothing is copied
            (void)mremap(P.stash + at, x.second, x.second, MREMAP_MAYMOVE | MREMAP_FIXED, x.first);
            at += x.second;
        }
    P.stash = nullptr;
    P.stash_bytes = 0;
    P.m.unlock();
}

// (never destroyed: buffers may come back while the process ends)
Pool &pool() {
    static Pool *p = [] {
        Pool *q = new Pool();
        pthread_atfork(before_fork, after_fork_parent, after_fork_child);
        return q;
    }();
    return *p;
}

// idle buffers, the largest first, until `bytes` more fit (m held; throws before it takes any)
void trim(Pool &P, size_t bytes, std::vector<void *> &gone) {
    if (P.bytes + bytes > kPoolBytes) gone.reserve(P.idle.size());
    while (!P.idle.empty() && P.bytes + bytes > kPoolBytes) {
        const auto it = std::prev(P.idle.end());
        gone.push_back(it->second);
        P.bytes -= it->first;
        P.idle.erase(it);
    }
}

void unpin(const std::vector<void *> &gone) {
    for (void *p : gone) (void)hipHostFree(p);
}

// whether [p, p + bytes) lies in a buffer handed out
bool pooled(const void *p, size_t bytes) {
    Pool &P = pool();
    std::lock_guard<std::mutex> g(P.m);
    auto it = P.out.upper_bound(const_cast<void *>(p));
    if (it == P.out.begin()) return false;
    --it;
    const char *a = static_cast<const char *>(it->first), *b = static_cast<const char *>(p);
    return b + bytes <= a + it->second;
}

void *acquire_or_throw(size_t bytes) {
    Pool &P = pool();
    bytes = (bytes + kGrain - 1) / kGrain * kGrain;
    if (bytes == 0 || bytes > kPoolBytes) return nullptr;
    std::vector<void *> gone;
    void *p = nullptr;
    {
        std::lock_guard<std::mutex> g(P.m);
        if (P.users == 0 || P.forked) return nullptr;
        auto it = P.idle.lower_bound(bytes);
        if (it != P.idle.end() && it->first <= bytes + bytes / 2) {
            p = it->second;
            P.out[p] = it->first;
            P.idle.erase(it);
            return p;
        }
        trim(P, bytes, gone);
        if (P.bytes + bytes <= kPoolBytes) P.bytes += bytes;   // reserved
        else bytes = 0;
    }
    unpin(gone);
    if (bytes == 0) return nullptr;
    const bool ok = hipHostMalloc(&p, bytes, hipHostMallocPortable) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    std::lock_guard<std::mutex> g(P.m);
    if (!ok) {
        P.bytes -= bytes;
        return nullptr;
    }
    try {
        P.out[p] = bytes;
    } catch (...) {
        P.bytes -= bytes;
        (void)hipHostFree(p);
        return nullptr;
    }
    return p;
}

// (null as well where the host has no memory for the pool's own records)
void *acquire(size_t bytes) noexcept {
    try {
        return acquire_or_throw(bytes);
    } catch (...) {
        return nullptr;
    }
}

void release_buffer(void *p) {
    Pool &P = pool();
    {
        std::lock_guard<std::mutex> g(P.m);
        const auto it = P.out.find(p);
        if (it == P.out.end()) return;
        const size_t bytes = it->second;
        P.out.erase(it);
        if (P.forked) {
            munmap(p, bytes);
            return;
        }
        if (P.users > 0) {
            try {
                P.idle.emplace(bytes, p);
                return;
            } catch (...) {
            }
        }
        P.bytes -= bytes;
    }
    (void)hipHostFree(p);
}

}  // namespace

void host_pool_retain() {
    Pool &P = pool();
    std::lock_guard<std::mutex> g(P.m);
    P.users += 1;
}

void host_pool_release() {
    Pool &P = pool();
    std::multimap<size_t, void *> gone;
    {
        std::lock_guard<std::mutex> g(P.m);
        if (--P.users > 0 || P.forked) return;
        gone.swap(P.idle);
        for (const auto &x : gone) P.bytes -= x.first;
    }
    for (const auto &x : gone) (void)hipHostFree(x.second);
}

int copy_out(const CopyOut *copies, int n, hipStream_t s) {
    size_t total = 0;
    bool pinned = true;
    for (int i = 0; i < n; ++i) {
        if (!copies[i].dst) continue;
        total += copies[i].bytes;
        pinned = pinned && pooled(copies[i].dst, copies[i].bytes);
    }
    if (total == 0) return TSI_OK;
    char *stage = !pinned && total <= kStageBytes ? static_cast<char *>(acquire(total)) : nullptr;
    if (!pinned && !stage) {
        // (these copies run on the null stream, which does not wait for the library's own streams)
        if (hipStreamSynchronize(s) != hipSuccess) return TSI_E_HIP;
        for (int i = 0; i < n; ++i)
            if (copies[i].dst &&
                hipMemcpy(copies[i].dst, copies[i].src, copies[i].bytes, hipMemcpyDeviceToHost) != hipSuccess)
                return TSI_E_HIP;
        return TSI_OK;
    }
    int rc = TSI_OK;
    size_t at = 0;
    for (int i = 0; i < n && rc == TSI_OK; ++i) {
        if (!copies[i].dst) continue;
        void *to = stage ? stage + at : copies[i].dst;
        if (hipMemcpyAsync(to, copies[i].src, copies[i].bytes, hipMemcpyDeviceToHost, s) != hipSuccess) rc = TSI_E_HIP;
        at += copies[i].bytes;
    }
    if (hipStreamSynchronize(s) != hipSuccess) rc = TSI_E_HIP;
    at = 0;
    for (int i = 0; i < n && rc == TSI_OK && stage; ++i) {
        if (!copies[i].dst) continue;
        std::memcpy(copies[i].dst, stage + at, copies[i].bytes);
        at += copies[i].bytes;
    }
    if (stage) release_buffer(stage);
    return rc;
}

}  // namespace tsi

using namespace tsi;

extern "C" {

void *tsi_host_buffer(size_t bytes) {
    return acquire(bytes);
}

void tsi_host_buffer_free(void *p) {
    if (p) release_buffer(p);
}

}  // extern "C"

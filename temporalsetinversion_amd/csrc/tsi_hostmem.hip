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
#include "tsi_hostmem.h"

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
};

// (never destroyed: buffers may come back while the process ends)
Pool &pool() {
    static Pool *p = new Pool();
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
        if (P.users == 0) return nullptr;
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
        if (--P.users > 0) return;
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

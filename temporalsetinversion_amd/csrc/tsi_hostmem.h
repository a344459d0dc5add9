// tsi_hostmem.h -- pinned host memory for what frames hand back (tsi_host_buffer), and copies out.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace tsi {

// Contexts and batches alive: the idle buffers of the pool are given back with the last of them.
void host_pool_retain();
void host_pool_release();
struct HostPoolUser {
    HostPoolUser() { host_pool_retain(); }
    ~HostPoolUser() { host_pool_release(); }
    HostPoolUser(const HostPoolUser &) = delete;
    HostPoolUser &operator=(const HostPoolUser &) = delete;
};

struct CopyOut {
    void *dst;         // null: not wanted
    const void *src;   // device
    size_t bytes;
};
// Device to host, after the work queued on s; complete on return.
int copy_out(const CopyOut *copies, int n, hipStream_t s);

}  // namespace tsi

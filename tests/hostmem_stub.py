"""tsi_hostmem.hip built for the CPU: a HIP runtime of the few calls it makes, whose streams run what is
queued on them only when they are waited for, and which does not order the null stream's copies
after them (the library's streams are non-blocking).  allocations() counts down to a failure of
operator new outside these calls (negative: never).  A driver's main() is compiled in."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "temporalsetinversion_amd")

RUNTIME = r"""
#pragma once
#include <sys/mman.h>
#include <cstddef>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <cstdlib>
#include <vector>
inline int &allocations() { static int n = -1; return n; }
struct Allocating {   // operator new does not fail while one lives
    int n = allocations();
    Allocating() { allocations() = -1; }
    ~Allocating() { allocations() = n; }
};
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorOutOfMemory = 2;
enum hipMemcpyKind { hipMemcpyDeviceToHost };
constexpr unsigned hipHostMallocPortable = 1u;
struct Stream { std::vector<std::function<void()>> queue; };
typedef Stream *hipStream_t;
inline size_t &pinned_bytes() { static size_t n = 0; return n; }
inline std::mutex &pinned_mutex() { static std::mutex m; return m; }
inline std::map<void *, size_t> &pinned() { static std::map<void *, size_t> m; return m; }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    Allocating allocating;
    st->queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
    Allocating allocating;
    for (auto &f : st->queue) f();
    st->queue.clear();
    return hipSuccess;
}
// pinned memory: a mapping that a forked child does not get, as the driver's
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    Allocating allocating;
    *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (*p == MAP_FAILED) return hipErrorOutOfMemory;
    madvise(*p, n, MADV_DONTFORK);
    std::lock_guard<std::mutex> g(pinned_mutex());
    pinned()[*p] = n;
    pinned_bytes() += n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    Allocating allocating;
    std::lock_guard<std::mutex> g(pinned_mutex());
    pinned_bytes() -= pinned()[p];
    munmap(p, pinned()[p]);
    pinned().erase(p);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

NEW = r"""
void *operator new(size_t n) {
    if (allocations() == 0) throw std::bad_alloc();
    if (allocations() > 0) allocations() -= 1;
    void *p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
"""


def build(tmp_path, main: str) -> str:
    """The driver's executable (main: C++ with a main(), tsi_hostmem.h and tsi.h included)."""
    inc = tmp_path / "hip"
    inc.mkdir()
    (inc / "hip_runtime.h").write_text(RUNTIME)
    src = tmp_path / "driver.cpp"
    hostmem = os.path.join(PKG, "csrc", "tsi_hostmem.hip")
    src.write_text(f'#include "{hostmem}"\n#include <cstdio>\n' + NEW + main)
    exe = str(tmp_path / "driver")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", str(tmp_path), "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(PKG, "csrc"), str(src), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def run(exe: str, *args: str) -> str:
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}{r.stderr}"
    return r.stdout

// tsi_kernels.hip -- CDNA4 (gfx950) kernels of the temporal set-inversion path.
//
// The reference runs one persistent WGSL kernel fed by a lock-free broker queue, one
// parent voxel per 8-thread workgroup, with every lane keeping a private 131 KB tape in
// global memory (compute.wgsl:3513-4056).  Here one frame is a fixed sequence of launches
// over a level-synchronous frontier:
//   k_frame_begin            seed the root (buf_main / first-frame seeding)
//   k_eval x levels          one 64-lane wavefront = 8 parents x 8 child octants; the tape
//                            is interpreted wave-uniformly (instructions via scalar loads,
//                            live values in a uniformly indexed VGPR file), then the cell is
//                            classified; subdivision / dealloc outputs are compacted with
//                            wavefront ballots + one atomic per wave and list
//   k_dealloc                the end of the dealloc cascade of compute.wgsl:3533-3543 / 4036-4044
//   k_frame_end              free-list merge, commit
// Frontier lists are split by whether the children will need the reverse pass, so the
// forward-only kernel carries no reverse-mode code or stack traffic.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "tsi.h"
#include "tsi_eval.h"
#include "tsi_interp.h"
#include "tsi_launch.h"

namespace tsi {

// ---------------------------------------------------------------- frame kernels

// One level with the interpreter (eval_level, tsi_eval.h), both lists side by side as in the compiled
// level kernel (a launch per list: 10 us more a level, of 110).
__global__ void __launch_bounds__(256) k_eval(KArgs a, int level, float time) {
    const uint32_t nb = gridDim.x, b = blockIdx.x, w = threadIdx.x >> 6, bwave = b * 4u + w;
    const uint32_t nf = __builtin_amdgcn_readfirstlane(level_split(a, level, nb));
    if (b < nf) eval_level<false, InterpEngine>(a, level, time, bwave, nf * 4u, bwave);
    else eval_level<true, InterpEngine>(a, level, time, (b - nf) * 4u + w, (nb - nf) * 4u, bwave);
}

__global__ void k_frame_begin(KArgs a) { frame_begin(a, threadIdx.x, blockDim.x); }

// The speculative pass's node list (spec_gather, tsi_eval.h): one block.
__global__ void __launch_bounds__(1024) k_spec_gather(KArgs a) { spec_gather(a, threadIdx.x, blockDim.x); }

// The interpreter's programs of a level, both lists (blockIdx.y): for each group of 8 entries the records
// that some entry's liveness record keeps, forward and reverse, with each entry's decisions.  Groups with an
// entry lacking a record run the full program.
__global__ void __launch_bounds__(256) k_prune(KArgs a, int level) {
    const int which = int(blockIdx.y);
    Counters *cnt = a.cnt;
    const uint32_t count = min(cnt->level[level].list[which], a.list_cap);
    if (count == 0) return;
    const uint32_t lane = lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t *prec = a.prune_rec[level & 1][which];
    uint32_t *desc = a.gdesc[which];
    const uint32_t nc = a.nchunks, cap = a.prune_cap;
    const uint32_t ngroups = (count + 7u) / 8u;
    const uint32_t *ffull = reinterpret_cast<const uint32_t *>(a.fprog);
    const uint32_t *rfull = reinterpret_cast<const uint32_t *>(a.rprog);
    for (uint32_t g = wave; g < ngroups; g += nwaves) {
        const uint32_t e0 = g * 8u;
        const uint32_t ne = count - e0 < 8u ? count - e0 : 8u;
        if (e0 + ne > a.prune_cap) {
            if (lane == 0) { desc[2u * g] = 0u; desc[2u * g + 1u] = 0u; }
            continue;
        }
        // union of the entries' live words; lane t holds chunks t and t + 64
        uint32_t u0 = 0, u1 = 0;
        const uint32_t c0 = lane, c1 = lane + 64u;
        for (uint32_t i = 0; i < ne; ++i) {
            const uint32_t *r = prec + size_t(kRecHead) * cap + e0 + i;
            if (c0 < nc) u0 |= r[size_t(c0) * cap];
            if (c1 < nc) u1 |= r[size_t(c1) * cap];
        }
        // exclusive prefix of per-chunk record counts, in chunk order
        const uint32_t n0 = __popc(u0), n1 = __popc(u1);
        uint32_t s0 = n0, s1 = n1;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y0 = uint32_t(__shfl_up(int(s0), off, 64)), y1 = uint32_t(__shfl_up(int(s1), off, 64));
            if (lane >= uint32_t(off)) { s0 += y0; s1 += y1; }
        }
        const uint32_t tot0 = bcast(s0, 63), tot1 = bcast(s1, 63);
        const uint32_t m = tot0 + tot1;
        const uint32_t off0 = s0 - n0, off1 = tot0 + s1 - n1;
        const uint32_t pad = program_stride(m);
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&cnt->level[level].pool_used, 2u * pad);
        base = bcast(base, 0);
        if (base + 2u * pad > a.pool_cap) {
            if (lane == 0) { desc[2u * g] = 0u; desc[2u * g + 1u] = 0u; }
            continue;
        }
        uint32_t *fw = reinterpret_cast<uint32_t *>(a.pool + base);
        uint32_t *rw = reinterpret_cast<uint32_t *>(a.pool + base + pad);
        for (int half = 0; half < 2; ++half) {
            const uint32_t c = half ? c1 : c0;
            uint32_t u = half ? u1 : u0, at = half ? off1 : off0;
            if (c >= nc) continue;
            uint32_t Lw[8], Rw[8], Vw[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                const uint32_t *r = prec + size_t(kRecHead + c) * cap + e0 + (i < ne ? i : 0u);
                Vw[i] = i < ne ? r[0] : 0u;
                Lw[i] = i < ne ? r[size_t(nc) * cap] : 0u;
                Rw[i] = i < ne ? r[size_t(2u * nc) * cap] : 0u;
            }
            while (u) {
                const uint32_t b = __builtin_ctz(u);
                u &= u - 1u;
                const uint32_t k = c * 32u + b;
                uint32_t modes = 0;
#pragma unroll
                for (uint32_t i = 0; i < 8; ++i) {
                    const uint32_t live = (Vw[i] >> b) & 1u;
                    const uint32_t md = live ? (((Lw[i] >> b) & 1u) | (((Rw[i] >> b) & 1u) << 1)) : 3u;
                    modes |= md << (2u * i);
                }
                const uint32_t *f = ffull + size_t(k) * 4u;
                uint32_t *fo = fw + size_t(at) * 4u;
                fo[0] = f[0];
                fo[1] = f[1];
                fo[2] = f[2];
                fo[3] = (f[3] & 0xFFFFu) | (modes << 16);
                const uint32_t *rr = rfull + size_t(a.nfwd - 1u - k) * 4u;
                uint32_t *ro = rw + size_t(m - 1u - at) * 4u;
                ro[0] = rr[0];
                ro[1] = rr[1];
                ro[2] = rr[2];
                ro[3] = (rr[3] & 0xFFFFu) | (modes << 16);
                ++at;
            }
        }
        // zero padding records after both programs (the interpreter prefetches past the end)
        for (uint32_t i = m * 4u + lane; i < pad * 4u; i += 64u) {
            fw[i] = 0u;
            rw[i] = 0u;
        }
        if (lane == 0) { desc[2u * g] = base; desc[2u * g + 1u] = m; }
    }
}

// The dealloc cascade's steps after the last level (dealloc_tail, tsi_eval.h).
__global__ void __launch_bounds__(256) k_dealloc(KArgs a, int step) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    LevelTally tl;
    tl.freed = dealloc_tail(a, step, wave, nwaves);
    if (tl.freed) flush_tally(a.tally, tl);
}

// The end of a frame: free-list merge (frame_end, tsi_eval.h) and, by the block that finishes last,
// the commit of the counters and the copy of what the host reads, into its memory (out).
// A launch and a copy kernel less than apart: 10 us of a frame's 300 at 256 x 256.
__global__ void __launch_bounds__(256) k_frame_end(KArgs a, CounterHead *out) {
    __shared__ uint32_t last;
    frame_end(a, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        last = atomicAdd(&a.cnt->finished, 1u) == gridDim.x - 1u;
    }
    __syncthreads();
    if (!last || threadIdx.x >= 64u) return;
    __threadfence();
    frame_commit(a);
    if (threadIdx.x == 0) a.cnt->finished = 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");   // the lanes' writes, for the copy
    const uint32_t *from = reinterpret_cast<const uint32_t *>(a.cnt);
    for (uint32_t i = threadIdx.x; i < uint32_t(sizeof(CounterHead) / 4u); i += 64u) reinterpret_cast<uint32_t *>(out)[i] = from[i];
}
__global__ void k_clear_nodes(KArgs a, uint64_t n) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
        a.st[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

__global__ void k_reset(KArgs a, float x0, float y0, float z0, float x1, float y1, float z1) {
    Counters *c = a.cnt;
    a.st[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   // main.rs:749-763: f=0, t=0, no children
    a.blo[0] = make_float4(x0, y0, z0, 0.0f);
    a.bhi[0] = make_float4(x1, y1, z1, 0.0f);
    a.grad[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    c->root_pending = 1;
    c->alloc_tickets = 0;
    c->free_top = 0;
    c->bump = 0;
    c->pending = 0;
    c->error = 0;
    c->frame_error = 0;
}

__global__ void k_enqueue_root(KArgs a) { a.cnt->root_pending = 1; }

// ---------------------------------------------------------------- frame dump

// RGBA32F -> RGBA8 as the reference's frame dump converts it (src/main.rs:709-711, image 0.24
// into_rgba8): clamp to [0, 1], scale by 255, round half away from zero.
__global__ void __launch_bounds__(256) k_rgba8(const float4 *in, uchar4 *out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = in[i];
    auto q = [](float x) -> unsigned char {
        return (unsigned char)roundf(wmin(wmax(x, 0.0f), 1.0f) * 255.0f);
    };
    out[i] = make_uchar4(q(v.x), q(v.y), q(v.z), q(v.w));
}

// ---------------------------------------------------------------- launchers

int launch_rgba8(const float4 *in, uchar4 *out, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_rgba8, dim3((n + 255u) / 256u), dim3(256), 0, s, in, out, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Blocks (4 wavefronts, 8 entries each) a list of level d can fill: it holds at most the 8^d nodes
// at depth d (and its dealloc list as many blocks), so the top levels launch a few blocks instead
// of the full grid (whose idle blocks would wait for dispatch behind a trace running beside).
uint32_t level_blocks(int d, uint32_t full) {
    if (d >= 7) return full;
    const uint64_t nodes = uint64_t(1) << (3 * d);
    const uint64_t groups = (nodes + 7u) / 8u;
    const uint64_t blocks = (groups + 3u) / 4u;
    return blocks < full ? uint32_t(blocks) : full;
}

int launch_frame(const KArgs &a, const FrameLaunch &fl, hipStream_t s, hipEvent_t e_eval0, hipEvent_t e_eval1,
                 const hipEvent_t *e_level) {
    const SpecLaunch *sp = fl.tape_eval ? fl.spec : nullptr;
    if (sp) {   // the speculative pass, beside the previous frame's last levels
        if (sp->wait) hipStreamWaitEvent(sp->stream, sp->wait, 0);
        hipLaunchKernelGGL(k_spec_gather, dim3(1), dim3(1024), 0, sp->stream, sp->args);
        hipEventRecord(sp->begin, sp->stream);   // times the tape kernel's launch only
        KArgs ka = sp->args;
        int level = -1;
        float t = fl.time;
        void *args[] = {&ka, &level, &t};
        if (hipModuleLaunchKernel((hipFunction_t)fl.tape_eval, sp->blocks, 1, 1, 256, 1, 1, 0, sp->stream, args,
                                  nullptr) != hipSuccess)
            return -1;
        hipEventRecord(sp->done, sp->stream);
    }
    hipLaunchKernelGGL(k_frame_begin, dim3(1), dim3(256), 0, s, a);
    if (sp) hipStreamWaitEvent(s, sp->done, 0);
    if (e_eval0) hipEventRecord(e_eval0, s);
    for (int d = 0; d < fl.levels; ++d) {
        const bool compiled = fl.tape_eval != nullptr;
        if (e_level) hipEventRecord(e_level[2 * d], s);
        if (a.prune && d > 0 && !compiled) {   // the interpreter's group programs
            hipLaunchKernelGGL(k_prune, dim3(fl.grid_misc, 2), dim3(256), 0, s, a, d);
        }
        // both lists of the level in one launch, which splits the grid: each list gets at least one block
        const uint32_t nb = std::min(fl.grid_fwd + fl.grid_rev, 2u * level_blocks(d, fl.grid_rev));
        if (compiled) {
            KArgs ka = a;
            int level = d;
            float t = fl.time;
            void *args[] = {&ka, &level, &t};
            if (hipModuleLaunchKernel((hipFunction_t)fl.tape_eval, nb, 1, 1, 256, 1, 1, 0, s, args, nullptr) !=
                hipSuccess)
                return -1;
        } else {
            hipLaunchKernelGGL(k_eval, dim3(nb), dim3(256), 0, s, a, d, fl.time);
        }
        if (e_level) hipEventRecord(e_level[2 * d + 1], s);
        if (sp && d == (sp->ready_level < fl.levels - 1 ? sp->ready_level : fl.levels - 1))
            hipEventRecord(sp->ready, s);
    }
    if (e_eval1) hipEventRecord(e_eval1, s);
    // levels 1..L-1 ran the cascade's steps 1..L-1 (eval_level); blocks dropped by the last
    // level and the descendants of earlier drops need at most two more
    hipLaunchKernelGGL(k_dealloc, dim3(fl.grid_misc), dim3(256), 0, s, a, fl.levels);
    hipLaunchKernelGGL(k_frame_end, dim3(64), dim3(256), 0, s, a, fl.out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_reset(const KArgs &a, const float box[6], uint64_t nodes, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_nodes, dim3(1024), dim3(256), 0, s, a, nodes);
    hipLaunchKernelGGL(k_reset, dim3(1), dim3(1), 0, s, a, box[0], box[1], box[2], box[3], box[4], box[5]);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_enqueue_root(const KArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_enqueue_root, dim3(1), dim3(1), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Copy of the nodes in use for an asynchronous trace; the count is read on the device (the
// host does not wait for the set inversion that produced it).
// (s_mask: the surface masks; s_grad: the gradients too, for gradient-normal shading; may be null)
__global__ void __launch_bounds__(256) k_snapshot(const Counters *cnt, const float4 *st, const float4 *blo,
                                                  const float4 *bhi, const float4 *grad, float4 *s_st, float4 *s_blo,
                                                  float4 *s_bhi, float4 *s_grad, uint32_t *s_mask, uint64_t nodes) {
    uint64_t used = (uint64_t(cnt->bump) + 1u) * 8u;
    if (used > nodes) used = nodes;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < used; i += uint64_t(gridDim.x) * blockDim.x) {
        s_st[i] = st[i];
        s_blo[i] = blo[i];
        s_bhi[i] = bhi[i];
        s_mask[i] = reinterpret_cast<const uint32_t *>(grad + i)[3];
        if (s_grad) s_grad[i] = grad[i];
    }
}

int launch_snapshot(const KArgs &a, float4 *s_st, float4 *s_blo, float4 *s_bhi, float4 *s_grad, uint32_t *s_mask,
                    uint64_t nodes, uint32_t grid, hipStream_t s) {
    hipLaunchKernelGGL(k_snapshot, dim3(grid), dim3(256), 0, s, a.cnt, a.st, a.blo, a.bhi, a.grad, s_st, s_blo, s_bhi,
                       s_grad, s_mask, nodes);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

int launch_fill_u32(uint32_t *p, uint32_t v, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u32, dim3((n + 255u) / 256u < 1024u ? (n + 255u) / 256u : 1024u), dim3(256), 0, s, p,
                       v, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tsi

// ---- check of the interval square root against the compiler's correctly rounded sqrtf ----

namespace tsi {

__global__ void __launch_bounds__(256) k_check_sqrt(uint32_t first, uint32_t count, unsigned long long *bad,
                                                    uint32_t *first_bad, uint32_t *done) {
    const uint32_t stride = gridDim.x * blockDim.x;   // count <= 2^31: i + stride never wraps
    uint32_t n = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride, ++n) {
        const uint32_t u = first + i;
        const float x = __uint_as_float(u);
        if (__float_as_uint(sqrt_nonneg(x)) != __float_as_uint(sqrtf(x))) {
            atomicAdd(bad, 1ull);
            atomicMin(first_bad, u);
        }
    }
    if (n) atomicAdd(done, n);
}

}  // namespace tsi

// Diagnostic export (no counterpart in the reference; not part of the tsi.h interface): compares
// sqrt_nonneg, the square root of SQRT_I, with sqrtf bit for bit for the binary32 values with bit
// patterns first .. first + count - 1 on the current device.  *mismatches receives the number of
// differences, *first_bad the smallest differing pattern (0xFFFFFFFF: none), *checked the number
// of values compared (count, when every thread ran).
extern "C" int tsi_check_sqrt(uint32_t first, uint32_t count, uint64_t *mismatches, uint32_t *first_bad,
                              uint32_t *checked) {
    if (!mismatches || !first_bad || !checked || count == 0 || count > 0x80000000u ||
        uint64_t(first) + count > (1ull << 32))
        return TSI_E_ARG;
    void *buf = nullptr;
    if (hipMalloc(&buf, 16) != hipSuccess) return TSI_E_OOM;
    unsigned long long *bad = static_cast<unsigned long long *>(buf);
    uint32_t *fb = reinterpret_cast<uint32_t *>(static_cast<char *>(buf) + 8);
    const uint32_t init[4] = {0u, 0u, 0xFFFFFFFFu, 0u};
    int rc = TSI_OK;
    if (hipMemcpy(buf, init, sizeof init, hipMemcpyHostToDevice) != hipSuccess) rc = TSI_E_HIP;
    if (rc == TSI_OK) {
        hipLaunchKernelGGL(tsi::k_check_sqrt, dim3(4096), dim3(256), 0, 0, first, count, bad, fb, fb + 1);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) rc = TSI_E_HIP;
    }
    uint32_t out[4] = {0u, 0u, 0u, 0u};
    if (rc == TSI_OK && hipMemcpy(out, buf, sizeof out, hipMemcpyDeviceToHost) != hipSuccess) rc = TSI_E_HIP;
    hipFree(buf);
    if (rc != TSI_OK) return rc;
    *mismatches = uint64_t(out[0]) | (uint64_t(out[1]) << 32);
    *first_bad = out[2];
    *checked = out[3];
    return TSI_OK;
}

// tsi_launch.h -- host-side launch sequences of the frame kernels (tsi_kernels.hip), for the
// runtime.  Kept apart from tsi_kernels.h, whose text is part of every generated tape kernel's
// source: a change here does not invalidate compiled tape kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "tsi.h"
#include "tsi_kernels.h"

namespace tsi {

// levels evaluated speculatively at frame start unless $TSI_SPEC_LEVELS says otherwise
constexpr long kSpecLevelsDefault = 7;

// every TSI_SHADE_* bit; tsi_params.shading with any other bit is rejected
constexpr uint32_t kShadeBits = TSI_SHADE_NORMALS | TSI_SHADE_GRADIENT | TSI_SHADE_CINEMATIC;

// The frame's speculative pass (KArgs::spec_*) on a stream of its own: it waits for `wait` (the
// previous frame's levels up to the deepest node it reads, or null), runs k_spec_gather and the
// level kernel at level -1 with `args` (its own saved-operand stack) on `blocks` blocks between
// `begin` and `done`; level 0 of the frame waits for `done`.  The frame records `ready` after
// its level `ready_level`, for the next frame's pass.
struct SpecLaunch {
    hipStream_t stream;
    hipEvent_t wait, begin, done, ready;
    KArgs args;
    uint32_t blocks;
    int ready_level;
};

struct FrameLaunch {
    int levels;
    float time;
    uint32_t grid_fwd, grid_rev, grid_misc;
    void *tape_eval;   // the tape's compiled level kernel (hipFunction_t), or null: k_eval
    const SpecLaunch *spec;   // or null
    CounterHead *out;         // host memory (pinned): the counters after the frame
};

// e_eval0 / e_eval1 (may be null) bracket the level loop; e_level (may be null) holds an event
// pair per level, recorded right before and after that level's evaluation launches.
int launch_frame(const KArgs &a, const FrameLaunch &fl, hipStream_t s, hipEvent_t e_eval0, hipEvent_t e_eval1,
                 const hipEvent_t *e_level);
int launch_reset(const KArgs &a, const float box[6], uint64_t nodes, hipStream_t s);
int launch_enqueue_root(const KArgs &a, hipStream_t s);
// A trace's frame.
struct TraceArgs {
    float view[16];
    uint32_t width, height;
    float time, zdist;
    float4 *rgba;
    float *depth;
    unsigned long long *visits; // kVisitSlots counters, kTallyStride words apart (one line each)
    uint32_t shading;           // TSI_SHADE_* (normal_viz, gradient normals, cinematic)
    const float4 *grad;         // the nodes' dx, dy, dz (gradient normals)
    const uint32_t *mask;       // the nodes' surface masks (grad[n].w), mask_stride words apart
    uint32_t mask_stride;
    uint32_t visit_slots;       // a power of two
    uint32_t stack;             // ray-stack entries: more than the octree's paths need, or the reference's 16
};

// claim counters of the persistent trace, each in a line of its own (2 * kTallyStride uint32 apart)
constexpr uint32_t kTraceQueues = 8;
// blocks > 0 (with next_quad, kTraceQueues counters zeroed on `s` before): the persistent form on that many
// blocks (k_trace_quads); else one block per tile (k_trace)
int launch_trace(const KArgs &a, const TraceArgs &t, hipStream_t s, uint32_t blocks = 0, uint32_t *next_quad = nullptr);
int launch_snapshot(const KArgs &a, float4 *s_st, float4 *s_blo, float4 *s_bhi, float4 *s_grad, uint32_t *s_mask,
                    uint64_t nodes, uint32_t grid, hipStream_t s);
int launch_rgba8(const float4 *in, uchar4 *out, uint32_t n, hipStream_t s);

// One frame of a batched trace (k_trace_batch): the session's nodes and the frame's arguments.
struct TraceJob {
    const float4 *st, *blo, *bhi, *grad;
    TraceArgs t;
    uint32_t blocks_x;  // blocks per row: ceil(width / side of a block's tile)
    uint32_t block0;    // the frame's first block in the launch
};
// (cinematic: every job's session shades with TSI_SHADE_CINEMATIC; no job mixes the two)
// stack: the largest of the jobs' TraceArgs::stack.
int launch_trace_batch(const TraceJob *jobs, uint32_t njobs, uint32_t total_blocks, bool cinematic, bool quads, uint32_t stack,
                       hipStream_t s);
// Whether a frame is traced with four lanes per ray (by its size; full launches only).
bool trace_quads(const TraceArgs &t);
bool trace_quads(uint64_t pixels, bool cinematic);
// Whether a full launch's grid holds the frame (else only the persistent form can trace it): its tiles are 4
// or 8 pixels high and the grid at most 65 535 of them, 262 140 or 524 280 rows of pixels.
bool trace_grid_fits(const TraceArgs &t);
// TraceArgs::stack for an octree whose nodes lie at depths up to `depth`.
uint32_t trace_stack_entries(int depth);
// After a trace (visits as in TraceArgs): the visits' sum to *out (pinned host memory), and the counters
// (n_clear words from visits on) cleared for the slot's next trace.
int launch_trace_end(unsigned long long *visits, uint32_t n_clear, unsigned long long *out, hipStream_t s);
// The canonical node records of an octree (tsi_read_nodes): every node reachable from the root
// through nodes with children, keyed by (depth, i, j, k).  Synchronous device reads.
int read_octree(const float4 *st_dev, const float4 *grad_dev, const Counters *cnt_dev, uint64_t nodes, tsi_node *out,
                uint64_t cap, uint64_t *count);
// Bytes that a chain's records (JitChain) may take on the current device: an eighth of what is free.  They
// only save work, and a program's own allocations after them would miss them.
uint64_t chain_memory();
// p[0 .. n) = v (a kernel, not a memset node, so that it also replays correctly in a captured graph)
int launch_fill_u32(uint32_t *p, uint32_t v, uint32_t n, hipStream_t s);

}  // namespace tsi

// tsi_trace.hip -- the octree ray traversal of rt_main / trace (compute.wgsl:4189-4403,
// 4650-4688) and the shading variants, for CDNA4.
//
// A traversal is one long dependent chain per ray (pop a node, set up a 2x2x2 DDA, step, load a
// child, test its box).  A frame of many rays is bound by the instructions of that chain, a frame of
// few by its latency, so the same code is written over two layouts of a ray's vectors:
//   LaneG  one lane per ray: the fewest instructions per ray;
//   QuadG  four lanes (a quad) per ray: lane k of the quad holds component k of every vector (x, y,
//          z; the fourth repeats z, so that quad-wide minima and maxima need no special case), and
//          sums, minima and broadcasts go through quad permutes, which are operands of ordinary
//          VALU instructions.  A chain's step issues about half the instructions, and 16 rays, not
//          64, wait for the slowest of them, at ~1.8 times the instructions for the frame.  The four
//          lanes compute every decision from the same values in the same order: a quad never
//          diverges.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "tsi.h"
#include "tsi_launch.h"
#include "tsi_wave.h"

namespace tsi {

namespace rays {

constexpr float kTrEps = 0.0001f;     // compute.wgsl:4140
constexpr float kDarken = 0.98f;      // compute.wgsl:3507
constexpr uint32_t kTraceThreads = 64;   // a wavefront: see k_trace
constexpr uint32_t kStackDepth = 16;  // compute.wgsl's stack: a push on a full one is dropped

// ---------------------------------------------------------------- layouts of a ray's vectors

struct V3 { float x, y, z; };
#define TSI_V3_OP(op)                                                                                        \
    TSI_DI V3 operator op(V3 a, V3 b) { return V3{a.x op b.x, a.y op b.y, a.z op b.z}; }                     \
    TSI_DI V3 operator op(V3 a, float b) { return V3{a.x op b, a.y op b, a.z op b}; }                        \
    TSI_DI V3 operator op(float a, V3 b) { return V3{a op b.x, a op b.y, a op b.z}; }
TSI_V3_OP(+)
TSI_V3_OP(-)
TSI_V3_OP(*)
TSI_V3_OP(/)
#undef TSI_V3_OP
TSI_DI V3 operator-(V3 a) { return V3{-a.x, -a.y, -a.z}; }

// operands of moderate size (walk's FAST form): magnitudes in [kMidLo, kMidHi]
constexpr float kMidLo = 0x1p-30f, kMidHi = 0x1p30f;
// three-operand minimum / maximum that return a NaN operand
TSI_DI float nmax(float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); }
TSI_DI float nmin(float a, float b, float c) { return __builtin_elementwise_minimum(__builtin_elementwise_minimum(a, b), c); }

TSI_DI float wsign(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }
// a negative component's step through the DDA grid: WGSL i32(sign(x))
TSI_DI int32_t step_of(float s) { return f2i_sat(s); }

struct LaneG {
    static constexpr uint32_t kLanes = 1u;
    typedef V3 V;
    struct IV { int32_t x, y, z; };
    static TSI_DI V pick(float x, float y, float z) { return V{x, y, z}; }
    static TSI_DI V load(const float4 *p, size_t n) { const float4 v = p[n]; return V{v.x, v.y, v.z}; }
    template <class F>
    static TSI_DI V map(V a, F f) { return V{f(a.x), f(a.y), f(a.z)}; }
    template <class F>
    static TSI_DI V map(V a, V b, F f) { return V{f(a.x, b.x), f(a.y, b.y), f(a.z, b.z)}; }
    template <class F>
    static TSI_DI V map(V a, V b, V c, F f) { return V{f(a.x, b.x, c.x), f(a.y, b.y, c.y), f(a.z, b.z, c.z)}; }
    static TSI_DI float maxc(V a) { return wmax(a.x, wmax(a.y, a.z)); }
    static TSI_DI float minc(V a) { return wmin(a.x, wmin(a.y, a.z)); }
    static TSI_DI float sum(V a) { return (a.x + a.y) + a.z; }
    static TSI_DI float x(V a) { return a.x; }
    static TSI_DI float y(V a) { return a.y; }
    static TSI_DI float z(V a) { return a.z; }
    static TSI_DI V cross(V a, V b) { return V{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
    static TSI_DI V swap_yz(V a) { return V{a.x, a.z, a.y}; }
    // grid position -> octant number mx + 2 my + 4 mz, and back
    static TSI_DI uint32_t octant_of(V m) {
        return uint32_t(f2i_sat(m.x)) + 2u * uint32_t(f2i_sat(m.y)) + 4u * uint32_t(f2i_sat(m.z));
    }
    static TSI_DI uint32_t octant_mid(V m) {   // |m| < 2^31
        return uint32_t(int32_t(m.x)) + 2u * uint32_t(int32_t(m.y)) + 4u * uint32_t(int32_t(m.z));
    }
    static TSI_DI V octant(uint32_t ci) { return V{float(ci & 1u), float((ci >> 1) & 1u), float((ci >> 2) & 1u)}; }
    // the steps of octant_of's number
    static TSI_DI IV steps(V s) { return IV{step_of(s.x), 2 * step_of(s.y), 4 * step_of(s.z)}; }
    static TSI_DI V fma(V a, V b, V c) {
        return V{__builtin_fmaf(a.x, b.x, c.x), __builtin_fmaf(a.y, b.y, c.y), __builtin_fmaf(a.z, b.z, c.z)};
    }
    // One DDA step along the axis whose side distance s is least: s moves by d there; len: |s - d|
    // after it, inc: the octant's change.  Returns whether several axes are least (no step is made
    // that the caller may use).  No NaN.
    static TSI_DI bool advance(V &s, V d, IV st, float &len, int32_t &inc) {
        const bool bx = s.x <= s.y && s.x <= s.z, by = s.y <= s.z && s.y <= s.x, bz = s.z <= s.x && s.z <= s.y;
        const V n = s + d, v = n - d;
        len = fabsf(bx ? v.x : (by ? v.y : v.z));
        inc = bx ? st.x : (by ? st.y : st.z);
        s = V{bx ? n.x : s.x, by ? n.y : s.y, bz ? n.z : s.z};
        return (bx && by) || (bz && (bx || by));
    }
    // the same decision, NaN as the reference's comparisons with minima have it
    static TSI_DI V least(V s, IV st, int32_t &inc) {
        const bool bx = s.x <= wmin(s.y, s.z), by = s.y <= wmin(s.z, s.x), bz = s.z <= wmin(s.x, s.y);
        inc = (bx ? st.x : 0) + (by ? st.y : 0) + (bz ? st.z : 0);
        return V{bx ? 1.0f : 0.0f, by ? 1.0f : 0.0f, bz ? 1.0f : 0.0f};
    }
    // whether every component's magnitude is in [kMidLo, kMidHi] (not, for a NaN)
    static TSI_DI bool mid(V a) { return mid(a, a, a); }
    static TSI_DI bool mid(V a, V b, V c) {
        const float hi = nmax(nmax(nmax(nmax(fabsf(a.x), fabsf(a.y), fabsf(a.z)), fabsf(b.x), fabsf(b.y)), fabsf(b.z), fabsf(c.x)),
                              fabsf(c.y), fabsf(c.z));
        const float lo = nmin(nmin(nmin(nmin(fabsf(a.x), fabsf(a.y), fabsf(a.z)), fabsf(b.x), fabsf(b.y)), fabsf(b.z), fabsf(c.x)),
                              fabsf(c.y), fabsf(c.z));
        return lo >= kMidLo && hi <= kMidHi;
    }

    // The ray's stack in LDS, one 8-byte entry per node of the path from the root: {children word,
    // surface mask | octant in its parent << 8}; boxes are read from the nodes.  walk_exact's
    // entries are {node, children word}.
    struct Stack {
        uint2 *base;   // entry 0 of this lane
        TSI_DI void put(uint32_t s, uint32_t node, uint32_t meta, V, V) const { base[s * kTraceThreads] = make_uint2(node, meta); }
        TSI_DI uint2 node(uint32_t s) const { return base[s * kTraceThreads]; }
        TSI_DI void box(const KArgs &a, uint32_t, uint32_t node, V &lo, V &hi) const {
            lo = load(a.blo, node);
            hi = load(a.bhi, node);
        }
        TSI_DI void put_box(uint32_t, V, V) const {}
        TSI_DI void put_node(uint32_t s, uint32_t meta, uint32_t mask) const { base[s * kTraceThreads] = make_uint2(meta, mask); }
        TSI_DI void get(const KArgs &a, uint32_t s, uint32_t &meta, uint32_t &mask, V &lo, V &hi) const {
            const uint2 e = base[s * kTraceThreads];
            const uint32_t up = base[(s == 0u ? 0u : s - 1u) * kTraceThreads].x;
            const uint32_t node = s == 0u ? 0u : (up - 1u) * 8u + (e.y >> 8);
            meta = e.x;
            mask = e.y;
            lo = load(a.blo, node);
            hi = load(a.bhi, node);
        }
    };
    static TSI_DI bool counts() { return true; }
    static TSI_DI void put_pixel(const TraceArgs &t, size_t pi, V c, float alpha, float depth) {
        t.rgba[pi] = make_float4(c.x, c.y, c.z, alpha);
        t.depth[pi] = depth;
    }
};

// quad permutes: lane k of each quad reads lane Pk
constexpr int quad_ctrl(int p0, int p1, int p2, int p3) { return p0 | (p1 << 2) | (p2 << 4) | (p3 << 6); }
template <int CTRL>
TSI_DI uint32_t qperm(uint32_t x) {
    return uint32_t(__builtin_amdgcn_mov_dpp(int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
TSI_DI float qperm(float x) { return __uint_as_float(qperm<CTRL>(__float_as_uint(x))); }
constexpr int kXor1 = quad_ctrl(1, 0, 3, 2), kXor2 = quad_ctrl(2, 3, 0, 1);
constexpr int kB0 = quad_ctrl(0, 0, 0, 0), kB1 = quad_ctrl(1, 1, 1, 1), kB2 = quad_ctrl(2, 2, 2, 2);
// the next axis and the one after it (the fourth lane repeats z)
constexpr int kNext = quad_ctrl(1, 2, 0, 0), kNext2 = quad_ctrl(2, 0, 1, 1);

struct QuadG {
    static constexpr uint32_t kLanes = 4u;
    typedef float V;
    typedef int32_t IV;
    static TSI_DI uint32_t axis() { return min(threadIdx.x & 3u, 2u); }
    static TSI_DI bool fourth() { return (threadIdx.x & 3u) == 3u; }
    static TSI_DI V pick(float x, float y, float z) { const uint32_t k = axis(); return k == 0u ? x : (k == 1u ? y : z); }
    static TSI_DI V load(const float4 *p, size_t n) { return reinterpret_cast<const float *>(p)[n * 4u + axis()]; }
    template <class F>
    static TSI_DI V map(V a, F f) { return f(a); }
    template <class F>
    static TSI_DI V map(V a, V b, F f) { return f(a, b); }
    template <class F>
    static TSI_DI V map(V a, V b, V c, F f) { return f(a, b, c); }
    // minimumNumber / maximumNumber are associative and commutative, and the repeated z changes
    // nothing: the values are those of min(x, min(y, z)) in any order
    static TSI_DI float maxc(V v) { v = wmax(v, qperm<kXor1>(v)); return wmax(v, qperm<kXor2>(v)); }
    static TSI_DI float minc(V v) { v = wmin(v, qperm<kXor1>(v)); return wmin(v, qperm<kXor2>(v)); }
    static TSI_DI float sum(V v) { return (x(v) + y(v)) + z(v); }
    static TSI_DI float x(V v) { return qperm<kB0>(v); }
    static TSI_DI float y(V v) { return qperm<kB1>(v); }
    static TSI_DI float z(V v) { return qperm<kB2>(v); }
    static TSI_DI V cross(V a, V b) { return qperm<kNext>(a) * qperm<kNext2>(b) - qperm<kNext2>(a) * qperm<kNext>(b); }
    static TSI_DI V swap_yz(V v) { return qperm<quad_ctrl(0, 2, 1, 1)>(v); }
    static TSI_DI uint32_t qadd(uint32_t v) { v = v + qperm<kXor1>(v); return v + qperm<kXor2>(v); }
    static TSI_DI uint32_t octant_of(V m) { return qadd(fourth() ? 0u : uint32_t(f2i_sat(m)) << axis()); }
    static TSI_DI uint32_t octant_mid(V m) { return qadd(fourth() ? 0u : uint32_t(int32_t(m)) << axis()); }
    static TSI_DI V octant(uint32_t ci) { return float((ci >> axis()) & 1u); }
    static TSI_DI IV steps(V s) { return fourth() ? 0 : step_of(s) * int32_t(1u << axis()); }
    static TSI_DI V fma(V a, V b, V c) { return __builtin_fmaf(a, b, c); }
    static TSI_DI bool advance(V &s, V d, IV st, float &len, int32_t &inc) {
        const float u = qperm<kNext>(s), w = qperm<kNext2>(s);   // (permutes read active lanes only: no short circuit)
        const bool b = s <= u && s <= w;
        const V n = s + d, v = n - d;
        len = maxc(b ? fabsf(v) : 0.0f);
        // the steps' sum (-7 .. 7) and their number, 4096 each
        const uint32_t k = qadd(b ? uint32_t(st) + (fourth() ? 0u : 4096u) : 0u);
        const uint32_t cnt = (k + 2048u) >> 12;
        inc = int32_t(k - (cnt << 12));
        s = b ? n : s;
        return cnt != 1u;
    }
    static TSI_DI V least(V s, IV st, int32_t &inc) {
        const bool b = s <= wmin(qperm<kNext>(s), qperm<kNext2>(s));
        inc = int32_t(qadd(b ? uint32_t(st) : 0u));
        return b ? 1.0f : 0.0f;
    }
    static TSI_DI bool all(bool p) {
        const uint32_t n = p ? 1u : 0u, m = n & qperm<kXor1>(n);
        return (m & qperm<kXor2>(m)) != 0u;
    }
    static TSI_DI bool mid(V a) { return mid(a, a, a); }
    static TSI_DI bool mid(V a, V b, V c) {
        return all(nmin(fabsf(a), fabsf(b), fabsf(c)) >= kMidLo && nmax(fabsf(a), fabsf(b), fabsf(c)) <= kMidHi);
    }

    // The ray's stack: entry s is 4 x 8 bytes of LDS, one per lane of the quad: {lo, hi} of the node's
    // stored box for the three axes, {children word, surface mask} (walk_exact: {node, children word})
    // in the fourth lane's, so that going back up the octree reads no node memory.
    struct Stack {
        uint2 *base;   // entry 0 of this lane
        TSI_DI void put(uint32_t s, uint32_t node, uint32_t meta, V lo, V hi) const {
            const bool w = fourth();
            base[s * kTraceThreads] = make_uint2(w ? node : __float_as_uint(lo), w ? meta : __float_as_uint(hi));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        TSI_DI uint2 node(uint32_t s) const { return base[s * kTraceThreads + 3u - (threadIdx.x & 3u)]; }
        TSI_DI void box(const KArgs &, uint32_t s, uint32_t, V &lo, V &hi) const {
            const uint2 b = base[int32_t(s * kTraceThreads) - (fourth() ? 1 : 0)];
            lo = __uint_as_float(b.x);
            hi = __uint_as_float(b.y);
        }
        TSI_DI void put_box(uint32_t s, V lo, V hi) const {
            if (!fourth()) base[s * kTraceThreads] = make_uint2(__float_as_uint(lo), __float_as_uint(hi));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        TSI_DI void put_node(uint32_t s, uint32_t meta, uint32_t mask) const {
            if (fourth()) base[s * kTraceThreads] = make_uint2(meta, mask);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        TSI_DI void get(const KArgs &a, uint32_t s, uint32_t &meta, uint32_t &mask, V &lo, V &hi) const {
            const uint2 e = node(s);
            meta = e.x;
            mask = e.y;
            box(a, s, 0u, lo, hi);
        }
    };
    static TSI_DI bool counts() { return (threadIdx.x & 3u) == 0u; }
    // colour components by the first three lanes, alpha by the fourth
    static TSI_DI void put_pixel(const TraceArgs &t, size_t pi, V c, float alpha, float depth) {
        const uint32_t k = threadIdx.x & 3u;
        reinterpret_cast<float *>(t.rgba)[pi * 4u + k] = k == 3u ? alpha : c;
        if (k == 0u) t.depth[pi] = depth;
    }
};

template <class G>
TSI_DI float gdot(typename G::V a, typename G::V b) { return G::sum(a * b); }
// (a sum of squares: +0 or more, +inf or NaN, where sqrt_nonneg equals sqrtf bit for bit)
template <class G>
TSI_DI float glength(typename G::V v) { return sqrt_nonneg(G::sum(v * v)); }
template <class G>
TSI_DI typename G::V gnormalize(typename G::V v) { return v / glength<G>(v); }   // v / length(v)

TSI_DI float mylerp(float a, float b, float t) {   // compute.wgsl:4116
    const float tt = wmin(wmax(t, 0.0f), 1.0f);
    return a * (1.0f - tt) + b * tt;
}

// efficient_slabs (compute.wgsl:4059-4070): whether the ray meets the box, and where
struct Slab { bool hit; float near_, far_; };
template <class G>
TSI_DI Slab slabs(typename G::V p0, typename G::V p1, typename G::V o, typename G::V inv) {
    const typename G::V t0 = (p0 - o) * inv, t1 = (p1 - o) * inv;
    const float d1 = G::maxc(G::map(t0, t1, [](float u, float v) { return wmin(u, v); }));
    const float d2 = G::minc(G::map(t0, t1, [](float u, float v) { return wmax(u, v); }));
    return Slab{d1 <= d2 && d2 >= 0.0f, wmax(d1, 0.0f), wmax(d2, 0.0f)};
}

// ---- division without its scaling steps ----
// The compiler's correctly rounded division scales its operands and fixes up zeros, infinities and
// NaN around a Newton-Raphson core; for operands of moderate size the core alone gives the same
// bits.  recip_mid: 1 / b for |b| in [2^-30, 2^30] (an exhaustive GPU test compares it with 1.0f / b);
// div_mid: a / b given r = recip_mid(b), by the core's two corrections, for |a| in [2^-90, 2^60]
// and |b| as above (every residual is then exact and no step under- or overflows).
TSI_DI float recip_mid(float b) {
    float y = __builtin_amdgcn_rcpf(b);
    y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
    return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}
TSI_DI float div_mid(float a, float b, float r) {
    float q = a * r;
    q = __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}
// The colour of a hit on leaf `leaf` (evaluated at time t_leaf) and normal_at_hit.  CIN: cinematic
// colouring (movement (0.7, 1e-4, 1e-4) fading to base 0.1, 4346-4374); the normal is
// finite_diff_normal's (1, 1, 1) for a tape scene, or the voxel's gradient with
// TSI_SHADE_GRADIENT (fast_normals = false, 4333-4342).  c: the colour so far, in every component.
template <class G, bool CIN>
TSI_DI typename G::V hit_colour(float c, float time, float t_leaf, uint32_t leaf, uint32_t shading, const float4 *grad,
                                typename G::V &nrm) {
    typedef typename G::V V;
    const bool normal_viz = (shading & TSI_SHADE_NORMALS) != 0;
    if (normal_viz || CIN) {
        V n = G::pick(1.0f, 1.0f, 1.0f);   // finite_diff_normal of a tape scene
        if (shading & TSI_SHADE_GRADIENT) n = G::load(grad, leaf);
        nrm = n;
        if (normal_viz) return gnormalize<G>(n * 1.0f) * 0.5f + 0.5f;   // 4333-4377
    }
    const float tt = (time - t_leaf) * 60.0f;
    if (CIN) {
        const float u = mylerp(1.0f - 0.0001f, 1.0f - 0.1f, tt);
        return c - G::pick(mylerp(1.0f - 0.7f, 1.0f - 0.1f, tt), u, u);
    }
    const float u = mylerp(1.0f, 0.0f, tt);
    return c - G::pick(mylerp(0.0f, 0.0f, tt), u, u);
}

TSI_DI float clamp01(float x) { return wmax(wmin(x, 1.0f), 0.0f); }

// trace (compute.wgsl:4189-4403) with its formulas as they stand.
template <class G, bool CIN>
TSI_DI void walk_exact(const KArgs &a, typename G::Stack stk, typename G::V ro, typename G::V rd,
                                        float time, typename G::V &col, float &dist, uint32_t &visits,
                                        uint32_t shading, const float4 *grad, uint32_t stack, typename G::V &nrm) {
    typedef typename G::V V;
    const bool normal_viz = (shading & TSI_SHADE_NORMALS) != 0;
    nrm = G::pick(0.0f, 0.0f, 0.0f);
    float c = 1.0f;    // the colour's three components until a hit
    V o2 = ro;
    bool intersected = false;
    const V inv = 1.0f / rd;
    // p0/p1: the box of the node being walked; q0/q1: its stored (unwidened) box, and qnode the node
    // that belongs to: a child's box is computed from it exactly as the set inversion computed the
    // stored one (lo + d * octant, d = (hi - lo) / 2; the product is exact, so the sum may be
    // fused), and children's boxes are not loaded
    V p0 = G::load(a.blo, 0), p1 = G::load(a.bhi, 0);
    V q0 = p0, q1 = p1;
    uint32_t qnode = 0u;
    uint32_t sp = 1;
    stk.put(0u, 0u, meta_of(a.st[0]) & kChildMask, q0, q1);
    Slab hit = slabs<G>(p0, p1, o2, inv);
    // back to the node on top of the stack
    auto ascend = [&]() {
        if (sp == 0u) return;
        qnode = stk.node(sp - 1u).x;
        stk.box(a, sp - 1u, qnode, q0, q1);
        p0 = q0;
        p1 = q1;
        hit = slabs<G>(p0, p1, o2, inv);
    };
    if (!hit.hit) sp = 0u;   // (the root is missed: the background)
    for (uint32_t iter = 0; iter < 5000u && sp != 0u; ++iter) {
        --sp;
        if (!hit.hit) {
            ascend();
            continue;
        }
        const uint2 top = stk.node(sp);
        const uint32_t region = top.x, rmeta = top.y;
        const V e = p1 - p0;
        const V r = ((o2 + (hit.near_ + kTrEps) * rd) - p0) * 2.0f / e;
        const V rdl = rd * (2.0f / e);
        const V m = G::map(r, [](float x) { return float(f2i_sat(floorf(x))); });
        const V dd = G::map(rdl, [](float x) { return 1.0f / fabsf(x); });
        const V sl = G::map(rdl, [](float x) { return wsign(x); });
        const typename G::IV st = G::steps(sl);
        V sd = ((sl * (m - r)) + sl * 0.5f + 0.5f) * dd;
        // mx + 2 my + 4 mz: all that the formulas use of the position
        uint32_t ci = G::octant_of(G::map(r, [](float x) { return floorf(x); }));
        V mk = G::pick(0.0f, 0.0f, 0.0f);
        const V old = o2;
        const float dark = !CIN && !normal_viz && G::maxc(e) < 1.0f ? kDarken : 1.0f;   // 4265
        // (after a DDA that left the 2x2x2 grid the popped node keeps the previous box, as in the
        // reference; its children's boxes are then loaded)
        const bool qown = qnode == region;
        const V h = (q1 - q0) / 2.0f;
        for (int i = 0; i < 32; ++i) {
            c = c * dark;
            const float t = (glength<G>(mk * (sd - dd)) + hit.near_) + kTrEps;
            o2 = old + t * rd;
            if (t >= hit.far_ - kTrEps) {
                o2 = old + hit.far_ * rd;
                ascend();
                break;
            }
            if (ci >= 8u) break;
            if (rmeta != 0u) {
                const uint32_t child = (rmeta - 1u) * 8u + ci;
                const float4 cs = a.st[child];
                ++visits;
                if (cs.x <= 0.0f) {
                    // the child's box as eval_level stored it (tsi_eval.h), from its parent's
                    const V oc = G::octant(ci);
                    V lo = G::fma(h, oc, q0), hi = G::fma(h, 1.0f + oc, q0);
                    if (!qown) {
                        lo = G::load(a.blo, child);
                        hi = G::load(a.bhi, child);
                    }
                    const Slab th = slabs<G>(lo - kTrEps, hi + kTrEps, o2, inv);
                    if (th.hit) {
                        const uint32_t cmeta = meta_of(cs) & kChildMask;
                        if (cmeta != 0u) {
                            // the walked node goes back on the stack (its entry is still there), then the child
                            ++sp;
                            if (sp < stack) {   // (TraceArgs::stack: full only where the reference's is)
                                stk.put(sp, child, cmeta, lo, hi);
                                ++sp;
                            }
                            p0 = lo - kTrEps;
                            p1 = hi + kTrEps;
                            q0 = lo;
                            q1 = hi;
                            qnode = child;
                            hit = th;
                            break;
                        }
                        intersected = true;
                        col = hit_colour<G, CIN>(c, time, cs.y, child, shading, grad, nrm);
                        break;
                    }
                }
            }
            int32_t inc;
            mk = G::least(sd, st, inc);
            sd = sd + mk * dd;
            ci = ci + uint32_t(inc);
        }
        if (intersected) break;
    }
    if (!intersected) col = G::pick(c, c, c);
    col = G::map(col, clamp01);
    dist = intersected ? fabsf(glength<G>(o2 - ro)) : -1.0f;
}

// Keeps a number a number, in a vector register (no instruction).
TSI_DI void in_vgpr(uint32_t &x) { asm volatile("" : "+v"(x)); }

// The same traversal, the same values bit for bit, for rays of moderate numbers; returns false where
// it cannot tell (walk_exact then takes the ray from its start).  What differs:
//   * divisions without their scaling steps (recip_mid, div_mid) while a node's box, the ray's
//     position in it and its grid direction are of moderate size; (A * 2) / e as A / (e / 2), an
//     exact rescaling;
//   * the distance of a DDA step, length(mask * (side - delta)), as |side - delta| of the one axis
//     stepped: the square root of a squared float is its magnitude while the square neither under-
//     nor overflows (side - delta is 0 or at least half an ulp of delta, and at most 33 delta); a
//     step of several axes at once goes to walk_exact;
//   * empty children are stepped over by the node's surface mask (grad[n].w: which children have
//     f <= 0, kept by eval_group), without a load; a child's children word and mask are loaded
//     when the ray enters it and first needed after the DDA set-up, so their latency is hidden,
//     and a leaf is recognised then;
//   * the stack is the path from the root: a node that goes back on it keeps its entry.
template <class G, bool CIN>
TSI_DI bool walk_fast(const KArgs &a, const TraceArgs &ta, typename G::Stack stk, typename G::V ro, typename G::V rd,
                      typename G::V &col, float &dist, uint32_t &visits, typename G::V &nrm) {
    typedef typename G::V V;
    const bool normal_viz = (ta.shading & TSI_SHADE_NORMALS) != 0;
    nrm = G::pick(0.0f, 0.0f, 0.0f);
    if (!G::mid(rd)) return false;
    const V inv = 1.0f / rd;
    const V sg = G::map(rd, [](float x) { return wsign(x); });
    const V sgh = sg * 0.5f;
    const typename G::IV st = G::steps(sg);
    float c = 1.0f;
    V o2 = ro;
    V p0 = G::load(a.blo, 0), p1 = G::load(a.bhi, 0);   // the walked box
    V q0 = p0, q1 = p1;                                 // the node's stored box
    uint32_t d = 0u;                                    // the node's depth: its entry on the stack
    uint32_t node = 0u;                                 // (of a node just entered)
    // (the stack's mask word: the surface mask, and above it the node's octant in its parent)
    uint32_t meta = meta_of(a.st[0]) & kChildMask, mask = ta.mask[0];
    // The walk's conditions are numbers in vector registers (in_vgpr): as conditions, each kept over
    // the divergent branches below takes three scalar instructions per change to merge, and a
    // wavefront issued nearly as many scalar instructions as vector ones (capsules at 512x512: 434
    // -> 348 us, at 1280x720 609 -> 465; path-traced csg at 960x540 9.7 -> 8.2 ms).
    uint32_t entered = 0u;       // the node was entered by the last iteration: it may be a leaf
    uint32_t own = 1u;           // p0/p1 are the node's (else the box of a node below, see walk_exact)
    uint32_t end = 0u;           // why the walk ended: it left (0), at a leaf (1), it cannot tell (2)
    float t_node = 0.0f;
    stk.put_box(0u, q0, q1);
    stk.put_node(0u, meta, mask);
    Slab hit = slabs<G>(p0, p1, o2, inv);
    uint32_t inside = hit.hit ? 1u : 0u;   // the walked box is hit
    if (inside != 0u) {
    for (uint32_t iter = 0; iter < 5000u; ++iter) {
        uint32_t way = 2u;       // 0: into a child, 1: back to the parent, 2: ... and to its box
        if (inside != 0u) {
            const V e = p1 - p0;
            const V eh = e * 0.5f;
            const V e2 = G::map(eh, recip_mid);       // 2 / e
            const V r = G::map((o2 + (hit.near_ + kTrEps) * rd) - p0, eh, e2, div_mid);
            const V rdl = rd * e2;
            const V m = G::map(r, [](float x) { return floorf(x); });
            const V dd = G::map(rdl, [](float x) { return recip_mid(fabsf(x)); });
            V sd = ((sg * (m - r)) + sgh + 0.5f) * dd;
            uint32_t ci = G::octant_mid(m);
            const float dark = !CIN && !normal_viz && G::maxc(e) < 1.0f ? kDarken : 1.0f;   // 4265
            const float leave = hit.far_ - kTrEps;
            const V h = (q1 - q0) * 0.5f;
            const bool ok = G::mid(eh, r, rdl) && G::minc(eh) > 0.0f;
            end = (entered != 0u && meta == 0u) ? 1u : (ok ? 0u : 2u);   // a leaf: the hit
            if (end != 0u) break;
            stk.put_node(d, meta, mask);
            entered = 0u;
            const V old = o2;
            // children that stop the march: those with a surface, and any number outside the grid
            const uint32_t stop = mask | 0xFFFFFF00u;
            float len = 0.0f, t;
            uint32_t steps = 0, tie = 0;
            way = 1u;
            for (;;) {
                for (;;) {
                    c = c * dark;
                    t = (len + hit.near_) + kTrEps;
                    const bool halt = t >= leave || ((stop >> min(ci, 31u)) & 1u) != 0u || steps == 32u;
                    if (halt) break;
                    ++steps;
                    int32_t inc;
                    tie = G::advance(sd, dd, st, len, inc) ? 1u : tie;
                    ci = ci + uint32_t(inc);
                }
                o2 = old + t * rd;
                if (t >= leave || ci >= 8u || (tie | (steps >> 5)) != 0u) break;
                ++steps;
                // the child's box as eval_level stored it (tsi_eval.h), from its parent's
                const V oc = G::octant(ci);
                V lo = G::fma(h, oc, q0), hi = G::fma(h, 1.0f + oc, q0);
                if (own == 0u) {
                    lo = G::load(a.blo, (meta - 1u) * 8u + ci);
                    hi = G::load(a.bhi, (meta - 1u) * 8u + ci);
                }
                const V w0 = lo - kTrEps, w1 = hi + kTrEps;
                const Slab th = slabs<G>(w0, w1, o2, inv);
                if (th.hit) {
                    way = 0u;
                    hit = th;
                    p0 = w0;
                    p1 = w1;
                    q0 = lo;
                    q1 = hi;
                    break;
                }
                int32_t inc;
                tie = G::advance(sd, dd, st, len, inc) ? 1u : tie;
                ci = ci + uint32_t(inc);
            }
            in_vgpr(way);
            in_vgpr(tie);
            visits += meta != 0u ? steps : 0u;
            end = (tie | (steps >> 5)) != 0u ? 2u : 0u;
            if (way == 0u) {
                node = (meta - 1u) * 8u + ci;
                meta = meta_of(a.st[node]) & kChildMask;
                t_node = a.st[node].y;
                mask = ta.mask[size_t(node) * ta.mask_stride] | (ci << 8);
                own = 1u;
                entered = 1u;
                ++d;
                if (d == ta.stack - 1u) end = 2u;   // (walk_exact knows what a full stack does)
                stk.put_box(d, q0, q1);
            } else if (t >= leave) {
                way = 2u;
                o2 = old + hit.far_ * rd;
            }
            if (end != 0u) break;
        }
        in_vgpr(way);
        if (way != 0u) {         // back to the parent
            if (d == 0u) break;
            --d;
            if (way == 2u) {
                stk.get(a, d, meta, mask, q0, q1);
                p0 = q0;
                p1 = q1;
                own = 1u;
                hit = slabs<G>(p0, p1, o2, inv);
                inside = hit.hit ? 1u : 0u;
            } else {
                V u, v;
                stk.get(a, d, meta, mask, u, v);
                own = 0u;
            }
        }
        in_vgpr(own);
        in_vgpr(inside);
        in_vgpr(entered);
    }
    }
    const bool ok = end != 2u;
    const bool intersected = end == 1u || (end == 0u && entered != 0u && meta == 0u);   // (or the iterations ended on a leaf)
    if (!ok) return false;
    col = G::pick(c, c, c);
    if (intersected) col = hit_colour<G, CIN>(c, ta.time, t_node, node, ta.shading, ta.grad, nrm);
    col = G::map(col, clamp01);   // (a ray that left keeps c in [0, 1])
    dist = intersected ? fabsf(glength<G>(o2 - ro)) : -1.0f;
    return true;
}

template <class G, bool CIN>
TSI_DI void trace_ray(const KArgs &a, const TraceArgs &ta, typename G::Stack stk, typename G::V ro, typename G::V rd,
                      typename G::V &col, float &dist, uint32_t &visits, typename G::V &nrm) {
    uint32_t n = 0;
    if (!walk_fast<G, CIN>(a, ta, stk, ro, rd, col, dist, n, nrm)) {
        n = 0;
        walk_exact<G, CIN>(a, stk, ro, rd, ta.time, col, dist, n, ta.shading, ta.grad, ta.stack, nrm);
    }
    visits += n;
}

// A pixel's ray direction in world space (ray_direction 4590-4594, view * vec4(d, 0) 4630) from
// its offsets on the image plane.
template <class G>
TSI_DI typename G::V ray_dir(const TraceArgs &t, float xyx, float xyy) {
    typedef typename G::V V;
    const float dx = xyx, dy = -xyy, dz = -t.zdist;
    const float len = sqrt_nonneg((dx * dx + dy * dy) + dz * dz);
    const V d = G::pick(dx, dy, dz) / len;
    const float *m = t.view;
    return ((G::pick(m[0], m[1], m[2]) * G::x(d) + G::pick(m[4], m[5], m[6]) * G::y(d)) +
            G::pick(m[8], m[9], m[10]) * G::z(d)) + G::pick(m[12], m[13], m[14]) * 0.0f;
}

// One pixel of rt_main (compute.wgsl:4650-4688): ray_direction, trace, get_color_single's normal_viz
// miss colour (4510-4514) and the 0.45 gamma.
template <class G>
TSI_DI void trace_pixel(const KArgs &a, const TraceArgs &t, uint32_t x, uint32_t y, typename G::Stack stk,
                        uint32_t &visits) {
    typedef typename G::V V;
    const float xyx = (float(x) - float(t.width) / 2.0f) + 0.5f;
    const float xyy = (float(y) - float(t.height) / 2.0f) + 0.5f;
    const V g = ray_dir<G>(t, xyx, xyy);
    const V eye = G::pick(t.view[12], t.view[13], t.view[14]);
    V c, n;
    float dist;
    trace_ray<G, false>(a, t, stk, eye, g, c, dist, visits, n);
    float ca = 1.0f;
    if ((t.shading & TSI_SHADE_NORMALS) && !(dist >= 0.0f)) {
        c = G::pick(10.0f, 10.0f, 10.0f);
        ca = 0.0f;
    }
    G::put_pixel(t, size_t(y) * t.width + x, G::map((0.0f + c) / 1.0f, [](float v) { return det_pow045(v); }),
                 (0.0f + ca) / 1.0f, dist);
}

// ---------------------------------------------------------------- cinematic shading

constexpr float kPiW = 3.14159274101257324f;   // compute.wgsl:2476 PI as f32

// frand0to1 (compute.wgsl:2466-2471): the LCG step seed * 747796405 + 1, then PCG's RXS-M-XS
// output permutation, mapped to [0, 1] by / 4294967295.0 (2^32 as f32); frand (2454-2459): [-1, 1].
TSI_DI float frand01(uint32_t &seed) {
    seed = seed * 747796405u + 1u;
    uint32_t w = ((seed >> ((seed >> 28u) + 4u)) ^ seed) * 277803737u;
    w = (w >> 22u) ^ w;
    return float(w) / 4294967295.0f;
}
TSI_DI float frand(uint32_t &seed) { return frand01(seed) * 2.0f - 1.0f; }

// getSampleBiased (4405-4434): a cosine-power lobe of exponent `power` around d
template <class G>
TSI_DI typename G::V sample_biased(typename G::V d, float power, uint32_t &seed) {
    typedef typename G::V V;
    const V dir = gnormalize<G>(d);
    const float dx = G::x(dir), dy = G::y(dir), dz = G::z(dir);
    const V ot = fabsf(dx) > fabsf(dz) ? G::pick(-dy, dx, 0.0f) : G::pick(0.0f, -dz, dy);   // ortho
    const V o1 = gnormalize<G>(ot);
    const V o2 = gnormalize<G>(G::cross(dir, o1));
    float rx = frand01(seed);
    float ry = frand01(seed);
    rx = rx * 2.0f * kPiW;
    ry = det_pow(ry, 1.0f / (power + 1.0f));
    const float om = sqrtf(1.0f - ry * ry);
    const float cx = det_cos(rx) * om, sy = det_sin(rx) * om;
    return (o1 * cx + o2 * sy) + dir * ry;
}

// fromSpherical (494-518)
template <class G>
TSI_DI typename G::V from_spherical(float px, float py) {
    return G::pick(det_cos(px) * det_sin(py), det_sin(px) * det_sin(py), det_cos(py));
}

// sunsky (520-640; Fragmentarium's Sunsky.frag) with turbidity = sunSize = 1 and the sky's sun
// intensity 1000 (423-427), RayleighPhase (429), totalMie (437), hgPhase (458), SunIntensity
// (478); pow(x, 2.0) is x * x.  The sun disk it computes is not in its result.
template <class G>
TSI_DI typename G::V sunsky(typename G::V view, float spx, float spy) {
    typedef typename G::V V;
    const float sadc = det_cos((1.0f * 3.1415927410125732f) / 180.0f);
    const V sd = gnormalize<G>(from_spherical<G>((spx - 0.0f) * 6.28000020980835f, (spy - 0.5f) * 3.140000104904175f));
    const V up = G::pick(0.0f, 0.0f, 1.0f);
    const float cvs = gdot<G>(view, sd);
    const float csu = gdot<G>(sd, up);
    const float cuv = gdot<G>(up, view);
    if (sadc == 1.0f) return G::pick(1.0f, 0.0f, 0.0f);
    const float sunE = 1000.0f * wmax(0.0f, 1.0f - det_exp(-((1.6110731611233942f - det_acos(csu)) / 1.5f)));
    const V ray = G::pick(5.176821105123963e-6f, 1.2785348189936485e-5f, 2.8530756026157178e-5f);
    // totalMie(lambda = (680, 550, 450) nm, K = (0.686, 0.678, 0.666), T = 1) * 0.005
    const float mc = (0.20000000298023224f * 1.0f) * 9.99999983775159e-18f;
    const float mk = (0.4339999854564667f * mc) * 3.1415927410125732f;
    const float tp = 2.0f * 3.1415927410125732f;
    const V q = G::pick(tp / 6.800000278417428e-7f, tp / 5.499999815583578e-7f, tp / 4.4999998749517545e-7f);
    const V mie = ((mk * (q * q)) * G::pick(0.6859999895095825f, 0.6779999732971191f, 0.6660000085830688f)) *
                      0.004999999888241291f;
    const float zen = wmax(0.0f, cuv);
    const float rol = 8400.0f / zen, mol = 1250.0f / zen;
    const V fex = G::map(-((ray * rol) + (mie * mol)), [](float v) { return det_exp(v); });
    const float rp = (3.0f / (16.0f * 3.1415927410125732f)) * (1.0f + cvs * cvs);
    const float g = 0.800000011920929f;
    const float hp = (1.0f / (4.0f * 3.1415927410125732f)) * ((1.0f - g * g) / det_pow((1.0f - (2.0f * g) * cvs) + g * g, 1.5f));
    const V lx = ray * rp + mie * hp;
    const V tl = ray + mie;
    const V se = sunE * (lx / tl);
    const float f = wmin(wmax(det_pow(1.0f - gdot<G>(up, sd), 5.0f), 0.0f), 1.0f);
    const V mx = 1.0f * (1.0f - f) + G::map(se * fex, [](float v) { return det_pow(v, 0.5f); }) * f;
    return ((se * (1.0f - fex)) * mx) * 0.009999999776482582f;
}

// LinearToSRGB (4600-4607) per channel, after clamping to [0, 1]
TSI_DI float linear_to_srgb(float x) {
    const float r = wmin(wmax(x, 0.0f), 1.0f);
    const float a = det_pow(r, 0.416666666666666667f) * 1.055f - 0.055f;
    const float b = r * 12.92f;
    const float t = r < 0.0031308f ? 1.0f : 0.0f;
    return a * (1.0f - t) + b * t;
}

// One pixel of rt_main with cinematic = true (compute.wgsl:4651-4688, 4620-4648, 4440-4523):
// seed3 from the pixel index and the time, 8 samples jittered by frand() * 0.5, each
// get_color_single's path of two bounces, each bounce a sun shadow ray (traced only when its
// result is read: sunlight > 0, 4501), a miss after the first bounce sees the sky; the mean goes
// through LinearToSRGB and the 0.45 gamma, alpha is the mean alpha.  The lighting is the
// scene-independent one (sun at (-0.1, 0.7), intensity 3, specular 1, albedo 1, sun size 0.01).
// Every ray of the pixel goes through the one trace_ray call below: a pixel's rays follow each
// other in a small state machine (sample, bounce, shadow), so a wavefront's pixels trace together
// wherever their paths are.  depth: the first sample's first ray.
template <class G>
TSI_DI void trace_pixel_cin(const KArgs &a, const TraceArgs &t, uint32_t x, uint32_t y, typename G::Stack stk,
                            uint32_t &visits) {
    typedef typename G::V V;
    constexpr float spx = -0.1f, spy = 0.7f, sun_i = 3.0f, specular_i = 1.0f, albedo = 1.0f, sunsize = 0.01f,
                    bgmul = 1.0f;
    const uint32_t pidx = y * t.width + x;
    uint32_t seed = pidx + uint32_t(12345.0f * (det_sin(t.time * 12345.0f) * 0.5f + 0.5f));
    const V eye = G::pick(t.view[12], t.view[13], t.view[14]);
    const V sundir = G::swap_yz(gnormalize<G>(from_spherical<G>((spx - 0.0f) * 6.28f, (spy - 0.5f) * 3.14f)));
    V acc = G::pick(0.0f, 0.0f, 0.0f);
    float aw = 0.0f;
    float depth0 = -1.0f;
    V frm = eye, dir = eye, lum = eye, direct = eye, old_rd = eye, nh = eye, ssd = eye;
    float sunlight = 0.0f;
    uint32_t sample = 0, bounce = 0;
    bool shadow = false;
    auto begin_sample = [&]() {
        const float jx = frand(seed);
        const float jy = frand(seed);
        const float px = float(x) + (jx * 1.0f) * 0.5f, py = float(y) + (jy * 1.0f) * 0.5f;
        const float xyx = (px - float(t.width) / 2.0f) + 0.5f;
        const float xyy = (py - float(t.height) / 2.0f) + 0.5f;
        dir = ray_dir<G>(t, xyx, xyy);
        frm = eye;
        lum = G::pick(1.0f, 1.0f, 1.0f);
        direct = G::pick(0.0f, 0.0f, 0.0f);
        bounce = 0;
        shadow = false;
    };
    begin_sample();
    for (uint32_t it = 0; it < 32u; ++it) {   // 8 samples x 2 bounces x (ray, shadow ray)
        V c, n;
        float d;
        trace_ray<G, true>(a, t, stk, frm, shadow ? ssd : dir, c, d, visits, n);
        bool end_bounce = false, end_sample = false;
        V res = G::pick(0.0f, 0.0f, 0.0f);
        float rw = 0.0f;
        if (shadow) {
            shadow = false;
            if (d < 0.0f) {   // not in shadow
                direct = direct + (lum * sunlight) * sun_i;
                const V half = gnormalize<G>(-old_rd + sundir);
                const float spec = (100.0f * det_pow(wmax(gdot<G>(nh, half), 0.0f), 30.0f)) * specular_i;
                direct = direct + lum * spec;
            }
            end_bounce = true;
        } else {
            if (sample == 0u && bounce == 0u) depth0 = d;
            if (d >= 0.0f) {
                const V hp = frm + dir * d;
                old_rd = dir;
                dir = sample_biased<G>(n, 3.0f, seed);
                lum = (lum * c) * albedo;
                frm = hp + n * 0.05f;
                const float j0 = frand(seed);
                const float j1 = frand(seed);
                const float j2 = frand(seed);
                ssd = gnormalize<G>(sundir + G::pick(j0, j1, j2) * sunsize);
                sunlight = gdot<G>(n, ssd);
                nh = n;
                if (sunlight > 0.0f) shadow = true;
                else end_bounce = true;
            } else if (bounce == 0u) {   // see_background = false (3506)
                res = G::pick(10.0f, 10.0f, 10.0f);
                rw = 0.0f;
                end_sample = true;
            } else {
                const V bg = sunsky<G>(G::swap_yz(dir), spx, spy);
                res = (direct + lum * bg) * bgmul;
                rw = 1.0f * bgmul;
                end_sample = true;
            }
        }
        if (end_bounce && ++bounce == 2u) {
            res = direct;
            rw = 1.0f;
            end_sample = true;
        }
        if (end_sample) {
            acc = acc + res;
            aw = aw + rw;
            if (++sample == 8u) break;
            begin_sample();
        }
    }
    acc = acc / 8.0f;
    aw = aw / 8.0f;
    G::put_pixel(t, size_t(pidx), G::map(acc, [](float v) { return det_pow045(linear_to_srgb(v)); }), aw, depth0);
}

// The wavefront's square tile of pixels at (x0, y0): 8x8 with one lane per ray, 4x4 with four
// (square tiles keep the rays of a wavefront close together, so that their traversals diverge less).
template <class G, bool CIN>
TSI_DI void shade_tile(const KArgs &a, const TraceArgs &t, uint32_t x0, uint32_t y0, typename G::Stack stk,
                       uint32_t &visits) {
    constexpr uint32_t side = G::kLanes == 1u ? 8u : 4u;
    const uint32_t r = (threadIdx.x & 63u) / G::kLanes;
    const uint32_t x = x0 + r % side, y = y0 + r / side;
    if (x >= t.width || y >= t.height) return;
    if (CIN) trace_pixel_cin<G>(a, t, x, y, stk, visits);
    else trace_pixel<G>(a, t, x, y, stk, visits);
}

template <class G>
TSI_DI void add_visits(const TraceArgs &t, uint32_t visits) {
    const uint64_t v = wave_sum64(G::counts() ? visits : 0u);
    const uint32_t slot = (blockIdx.x + blockIdx.y * 5u) & (t.visit_slots - 1u);
    if (lane_id() == 0 && v) atomicAdd((unsigned long long *)t.visits + slot * kTallyStride, (unsigned long long)v);
}

}  // namespace rays
using namespace rays;

// One wavefront per block: a block of four keeps its LDS (the ray stacks: 8 KB a wavefront) until its
// slowest wavefront is done, and with times of 40 to 110 us a SIMD held 1.9 wavefronts on average
// where 5 fit.
template <class G, bool CIN>
__global__ void __launch_bounds__(kTraceThreads) k_trace(KArgs a, TraceArgs t) {
    extern __shared__ uint2 stack_lds[];
    constexpr uint32_t side = G::kLanes == 1u ? 8u : 4u;
    uint32_t visits = 0;
    shade_tile<G, CIN>(a, t, blockIdx.x * side, blockIdx.y * side, typename G::Stack{stack_lds + threadIdx.x}, visits);
    add_visits<G>(t, visits);
}

// The same pixels on a grid of a few wavefronts per CU: each claims 8x8-pixel quadrants
// (row-major over the frame, dealt to kTraceQueues counters) until none is left.  A full launch keeps every CU's
// wave slots filled with trace wavefronts while any block is pending, so the next frame's level
// kernels, launched beside it, wait for slots; this leaves the CUs most of their slots.  Each pixel
// is shaded by the same code as in k_trace: the frame is the same.
template <bool CIN>
__global__ void __launch_bounds__(kTraceThreads) k_trace_quads(KArgs a, TraceArgs t, uint32_t *next_quad, uint32_t quads_x,
                                                     uint32_t nquads) {
    extern __shared__ uint2 stack_lds[];
    const uint32_t queue = blockIdx.x % kTraceQueues;
    uint32_t visits = 0;
    for (;;) {
        uint32_t q = 0;
        if (lane_id() == 0) q = atomicAdd(next_quad + queue * 2u * kTallyStride, 1u);
        q = __builtin_amdgcn_readfirstlane(q) * kTraceQueues + queue;
        if (q >= nquads) break;
        shade_tile<LaneG, CIN>(a, t, (q % quads_x) * 8u, (q / quads_x) * 8u, LaneG::Stack{stack_lds + threadIdx.x}, visits);
    }
    add_visits<LaneG>(t, visits);
}

// The frames of a batch in one launch: block i is a tile (shade_tile) of the frame whose blocks
// [jobs[j].block0, jobs[j + 1].block0) hold it, row-major over blocks_x blocks per row
// (a persistent grid taking tiles
// from a counter measured slower: a frame's slowest tiles then ran one after another in a few
// wavefronts, where the hardware dispatcher starts each block on the first free slot).
template <class G, bool CIN>
__global__ void __launch_bounds__(kTraceThreads) k_trace_batch(const TraceJob *jobs, uint32_t njobs) {
    extern __shared__ uint2 stack_lds[];
    const uint32_t blk = blockIdx.x;
    uint32_t lo = 0, hi = njobs;   // last job with block0 <= blk
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (as_const(jobs[mid]).block0 <= blk) lo = mid; else hi = mid;
    }
    // the job table is written before the launch and only read here: scalar loads (as_const)
    const auto &J = as_const(jobs[__builtin_amdgcn_readfirstlane(lo)]);
    KArgs a{};
    a.st = const_cast<float4 *>(J.st);
    a.blo = const_cast<float4 *>(J.blo);
    a.bhi = const_cast<float4 *>(J.bhi);
    TraceArgs t;
    for (int k = 0; k < 16; ++k) t.view[k] = J.t.view[k];
    t.width = J.t.width;
    t.height = J.t.height;
    t.time = J.t.time;
    t.zdist = J.t.zdist;
    t.rgba = J.t.rgba;
    t.depth = J.t.depth;
    t.visits = J.t.visits;
    t.shading = J.t.shading;
    t.grad = J.t.grad;
    t.mask = J.t.mask;
    t.mask_stride = J.t.mask_stride;
    t.visit_slots = J.t.visit_slots;
    t.stack = J.t.stack;
    const uint32_t local = blk - J.block0;
    constexpr uint32_t side = G::kLanes == 1u ? 8u : 4u;
    uint32_t visits = 0;
    shade_tile<G, CIN>(a, t, (local % J.blocks_x) * side, (local / J.blocks_x) * side,
                       typename G::Stack{stack_lds + threadIdx.x}, visits);
    add_visits<G>(t, visits);
}

// See launch_trace_end: one wavefront.  (A memset before the trace and a copy after it: 7 us more.)
__global__ void k_trace_end(unsigned long long *visits, uint32_t n_clear, unsigned long long *out) {
    const uint64_t v = wave_sum64(lane_id() < kVisitSlots ? visits[lane_id() * kTallyStride] : 0u);
    for (uint32_t i = lane_id(); i < n_clear; i += 64u) visits[i] = 0u;
    if (lane_id() == 0) *out = v;
}

// ---------------------------------------------------------------- launchers

int launch_trace_end(unsigned long long *visits, uint32_t n_clear, unsigned long long *out, hipStream_t s) {
    hipLaunchKernelGGL(k_trace_end, dim3(1), dim3(64), 0, s, visits, n_clear, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Frames (a batch's together) of at most this many pixels are traced with four lanes per ray: their wavefronts then
// still find free SIMDs, and the frame takes the latency of its longest chains, which are shorter so
// (64x48 spheres: 88 against 108 us; csg at 362x362: 296 against 307).  Larger frames are bound by
// instructions (448x448: capsules 382 against 327 us, csg 332 against 290, spheres 116 against 122).
// A batch of one frame of 320x240: 90 against 118 us.
// A path-traced pixel is 8 samples of up to 4 rays, chains so long that the line lies higher (csg at
// 641x361: 6.7 against 7.2 ms, capsules 7.1 against 8.2; at 960x540 9.2 against 8.0 and 9.1 against 8.8).
constexpr uint64_t kQuadPixels = 147456, kQuadPixelsCinematic = 393216;

// LDS of a wavefront's ray stacks: entries x 64 lanes x 8 B.
static uint32_t stack_bytes(uint32_t entries) { return entries * kTraceThreads * uint32_t(sizeof(uint2)); }

uint32_t trace_stack_entries(int depth) { return std::min(kStackDepth, uint32_t(depth) + 3u); }

int launch_trace_batch(const TraceJob *jobs, uint32_t njobs, uint32_t total_blocks, bool cinematic, bool quads, uint32_t stack,
                       hipStream_t s) {
    auto *k = quads ? (cinematic ? k_trace_batch<QuadG, true> : k_trace_batch<QuadG, false>)
                    : (cinematic ? k_trace_batch<LaneG, true> : k_trace_batch<LaneG, false>);
    hipLaunchKernelGGL(k, dim3(total_blocks), dim3(kTraceThreads), stack_bytes(stack), s, jobs, njobs);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

bool trace_quads(uint64_t pixels, bool cinematic) { return pixels <= (cinematic ? kQuadPixelsCinematic : kQuadPixels); }

bool trace_quads(const TraceArgs &t) {
    return trace_quads(uint64_t(t.width) * t.height, (t.shading & TSI_SHADE_CINEMATIC) != 0);
}

constexpr uint32_t kMaxGridRows = 65535;   // what a grid's second dimension may hold

// pixels of a side of a full launch's tile (shade_tile)
static uint32_t tile_of(bool quads) { return quads ? 4u : 8u; }

bool trace_grid_fits(const TraceArgs &t) {
    const uint32_t tile = tile_of(trace_quads(t));
    return t.height <= kMaxGridRows * tile;
}

int launch_trace(const KArgs &a, const TraceArgs &t, hipStream_t s, uint32_t blocks, uint32_t *next_quad) {
    const bool cin = (t.shading & TSI_SHADE_CINEMATIC) != 0;
    if (blocks && next_quad) {   // persistent: `blocks` blocks, *next_quad zeroed on the stream before
        const uint32_t qx = (t.width + 7u) / 8u, nq = qx * ((t.height + 7u) / 8u);
        const uint32_t nb = std::min(blocks, std::max(kTraceQueues, nq));   // (a block for every queue)
        if (cin) hipLaunchKernelGGL(k_trace_quads<true>, dim3(nb), dim3(kTraceThreads), stack_bytes(t.stack), s, a, t, next_quad, qx, nq);
        else hipLaunchKernelGGL(k_trace_quads<false>, dim3(nb), dim3(kTraceThreads), stack_bytes(t.stack), s, a, t, next_quad, qx, nq);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    const bool quad = trace_quads(t);
    const uint32_t tile = tile_of(quad);
    const dim3 grid((t.width + tile - 1u) / tile, (t.height + tile - 1u) / tile);
    if (quad) {
        if (cin) hipLaunchKernelGGL((k_trace<QuadG, true>), grid, dim3(kTraceThreads), stack_bytes(t.stack), s, a, t);
        else hipLaunchKernelGGL((k_trace<QuadG, false>), grid, dim3(kTraceThreads), stack_bytes(t.stack), s, a, t);
    } else {
        if (cin) hipLaunchKernelGGL((k_trace<LaneG, true>), grid, dim3(kTraceThreads), stack_bytes(t.stack), s, a, t);
        else hipLaunchKernelGGL((k_trace<LaneG, false>), grid, dim3(kTraceThreads), stack_bytes(t.stack), s, a, t);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tsi

// ---- check of the division core against the compiler's correctly rounded division ----

namespace tsi {

// recip: recip_mid(x) against 1.0f / x for the bit patterns first .. first + count - 1; otherwise
// count pseudo-random pairs (a splitmix64 stream from `first`) of moderate operands, div_mid
// against a / b.
__global__ void __launch_bounds__(256) k_check_div(uint32_t first, uint32_t count, bool recip, unsigned long long *bad,
                                                   uint32_t *first_bad, uint32_t *done) {
    const uint32_t stride = gridDim.x * blockDim.x;   // count <= 2^31: i + stride never wraps
    uint32_t n = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride, ++n) {
        bool same;
        if (recip) {
            const float x = __uint_as_float(first + i);
            same = __float_as_uint(recip_mid(x)) == __float_as_uint(1.0f / x);
        } else {
            uint64_t z = (uint64_t(first) << 32) + uint64_t(i) * 0x9E3779B97F4A7C15ull;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            // mantissas and sign from z; exponents of b in [-30, 29], of a in [-60, 59]
            const uint32_t ea = 67u + uint32_t((z >> 47) % 120u), eb = 97u + uint32_t((z >> 54) % 60u);
            const float a = __uint_as_float((uint32_t(z) & 0x807FFFFFu) | (ea << 23));
            const float b = __uint_as_float((uint32_t(z >> 24) & 0x007FFFFFu) | (eb << 23));
            same = __float_as_uint(div_mid(a, b, recip_mid(b))) == __float_as_uint(a / b);
        }
        if (!same) {
            atomicAdd(bad, 1ull);
            atomicMin(first_bad, first + i);
        }
    }
    if (n) atomicAdd(done, n);
}

}  // namespace tsi

// Diagnostic export (no counterpart in the reference; not part of the tsi.h interface): compares the
// trace's division core with the compiler's division bit for bit (k_check_div) on the current
// device.  *mismatches receives the number of differences, *first_bad the smallest differing
// index (0xFFFFFFFF: none), *checked the number of operations compared.
extern "C" int tsi_check_div(uint32_t first, uint32_t count, int32_t recip, uint64_t *mismatches, uint32_t *first_bad,
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
        hipLaunchKernelGGL(tsi::k_check_div, dim3(4096), dim3(256), 0, 0, first, count, recip != 0, bad, fb, fb + 1);
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

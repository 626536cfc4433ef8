// Closest-hit traversal of the quantised BVH4 and BVH8 (bvh.h) on gfx950: one ray per lane, the
// traversal stack in LDS (one column per lane, so the 64 lanes of a wave hit distinct banks),
// children near-to-far by a sort of integer keys, octant-selected slab planes (one byte permute
// per two planes, one mixed-precision FMA per plane).
//
// Result = Scene.trace_ray (include/merian-shaders/scene/scene.slang:62-76) with the ray query
// of acceleration-structure.slang:59-72: back-face culling per triangle, 8-bit instance mask,
// t in [tmin, tmax], ties at equal t to the lowest triangle id.
#pragma once

#include "bvh.h"
#include "mrt_device.h"
#include "mrt_kernels.h"

namespace mrt {

struct HitRec {
    uint32_t id; // global triangle id, 0xFFFFFFFF = miss
    float t, u, v;
};

// Textbook Moller-Trumbore (1997) in a fixed operation order; no contraction (the file is
// compiled with -ffp-contract=off), so CPU and GPU round identically.
__device__ __forceinline__ void test_triangle(const float4 A, const float4 B, const float4 Cc, f3 o, f3 d, float tmin,
                                              float tmax, uint32_t ray_mask, HitRec& best) {
    const uint32_t flags = __float_as_uint(B.w);
    if (((flags >> 8) & ray_mask) == 0u) return;
    const f3 e1{B.x, B.y, B.z}, e2{Cc.x, Cc.y, Cc.z};
    const f3 p = cross(d, e2);
    const float det = dot(e1, p);
    if (flags & 1u) {
        if (!(det > 0.0f)) return;
    } else {
        if (!(det != 0.0f)) return;
    }
    const float inv = 1.0f / det;
    const f3 s = o - f3{A.x, A.y, A.z};
    const float u = dot(s, p) * inv;
    if (!(u >= 0.0f && u <= 1.0f)) return;
    const f3 q = cross(s, e1);
    const float v = dot(d, q) * inv;
    if (!(v >= 0.0f && u + v <= 1.0f)) return;
    const float t = dot(e2, q) * inv;
    if (!(t >= tmin && t <= tmax)) return;
    const uint32_t id = __float_as_uint(A.w);
    if (t < best.t || (t == best.t && id < best.id)) best = HitRec{id, t, u, v};
}

constexpr uint32_t TRAVERSAL_DONE = 0xFFFFFFFFu;
constexpr int KEY_MISS = 0x7FFFFFFF; // sort key of a child whose box is missed: above every limit

// Work counters of one traversal (COUNT variant only): node visits and triangle tests.
struct TraversalCount {
    uint32_t nodes = 0, tris = 0;
};

// Traversal stack of one lane: the first TRACE_LDS_STACK entries in an LDS column (stride = threads
// per block, a compile-time constant, so a wave's 64 lanes touch 64 distinct banks), deeper entries
// in a per-lane column of a global overflow area (stride = threads of the grid). Near-first
// traversal rarely goes past the LDS part.
typedef __attribute__((address_space(3))) uint32_t* lds_u32;
typedef __attribute__((address_space(1))) uint32_t* global_u32;
struct LaneStack {
    uint32_t* lds; // this lane's column
    uint32_t* ovf;
    uint32_t ovf_stride;
};
// explicit address spaces keep LDS and overflow accesses apart (ds and global instructions rather
// than flat ones through a selected pointer)
__device__ __forceinline__ void stack_poke(const LaneStack& s, int i, uint32_t e) {
    if (i < TRACE_LDS_STACK) {
        ((lds_u32)s.lds)[i * TRACE_BLOCK] = e;
    } else {
        ((global_u32)s.ovf)[size_t(i - TRACE_LDS_STACK) * s.ovf_stride] = e;
    }
}
__device__ __forceinline__ void stack_push(const LaneStack& s, int& sp, uint32_t e) { stack_poke(s, sp++, e); }
__device__ __forceinline__ uint32_t stack_peek(const LaneStack& s, int i) {
    if (i < TRACE_LDS_STACK) return ((lds_u32)s.lds)[i * TRACE_BLOCK];
    return ((global_u32)s.ovf)[size_t(i - TRACE_LDS_STACK) * s.ovf_stride];
}

// Per-lane traversal state between steps.
struct RayState {
    f3 o, d;
    float ix, iy, iz, ox, oy, oz;
    float t0, tmin, tmax;
    int klim;     // far limit of the box tests (far_limit)
    uint32_t neg; // bit k: direction component k is negative
    uint32_t psel[3]; // v_perm selector per axis: the near planes of children 0 and 1 (lo for a
                      // positive direction, hi for a negative one) as two zero-extended bytes;
                      // + 0x00020002: children 2 and 3; swapped operands: the far planes
    HitRec best;
    int sp;
    uint32_t cur;  // next entry to process; TRAVERSAL_DONE when the stack is exhausted
    uint32_t leaf; // postponed leaf entry awaiting its triangle tests; TRAVERSAL_DONE when none
};

__device__ __forceinline__ bool is_inner(uint32_t e) { return !(e & LEAF_FLAG); }
__device__ __forceinline__ bool is_leaf(uint32_t e) { return e != TRAVERSAL_DONE && (e & LEAF_FLAG); }

// Far limit of the box tests: min(tmax, best.t) widened by 2 ulp. Octant order compares distances
// and takes the limit's bits as they are (upwards also from a negative one: an interval of one
// negative point keeps its boxes). Sorted order takes it as a sort key: a child is visited while its
// key is at most this. Keys compare as signed integers, so non-negative distances compare as they
// should and a negative one (a box around the origin of a ray with a negative tmin) is below every
// limit; a negative limit admits everything and leaves the rejection to the triangle test.
template <bool SORTED> __device__ __forceinline__ int far_limit(float tmax, float t) {
    const float m = fminf(tmax, t);
    if constexpr (!SORTED) return int(__float_as_uint(m + fabsf(m) * 2.4e-7f));
    const float lim = m * 1.00000024f;
    return lim >= 0.f ? int(__float_as_uint(fabsf(lim)) | 0xFFu) : KEY_MISS - 1; // fabsf: -0 is 0
}

// dir_min: smallest magnitude of a direction component in the box tests (DeviceScene.dir_min).
template <bool SORTED>
__device__ __forceinline__ void ray_begin(RayState& r, f3 o, f3 d, float tmin, float tmax, float dir_min) {
    r.o = o;
    r.d = d;
    const float dx = fabsf(d.x) < dir_min ? copysignf(dir_min, d.x) : d.x;
    const float dy = fabsf(d.y) < dir_min ? copysignf(dir_min, d.y) : d.y;
    const float dz = fabsf(d.z) < dir_min ? copysignf(dir_min, d.z) : d.z;
    // the hardware reciprocal (1 ulp) instead of a correctly rounded division: 1/d only feeds
    // the box tests, whose boxes the builder pads by extent/1024 + magnitude/65536, far above
    // an ulp of the slab distances; the triangle test uses d itself
    r.ix = __builtin_amdgcn_rcpf(dx);
    r.iy = __builtin_amdgcn_rcpf(dy);
    r.iz = __builtin_amdgcn_rcpf(dz);
    r.ox = o.x * r.ix;
    r.oy = o.y * r.iy;
    r.oz = o.z * r.iz;
    r.neg = (r.ix < 0.f ? 1u : 0u) | (r.iy < 0.f ? 2u : 0u) | (r.iz < 0.f ? 4u : 0u);
    r.tmin = tmin;
    r.tmax = tmax;
    r.t0 = tmin - fabsf(tmin) * 2.4e-7f;
    r.best = HitRec{TRAVERSAL_DONE, __builtin_inff(), 0.f, 0.f};
    r.klim = far_limit<SORTED>(tmax, r.best.t);
    r.psel[0] = (r.neg & 1u) ? 0x0C050C04u : 0x0C010C00u;
    r.psel[1] = (r.neg & 2u) ? 0x0C050C04u : 0x0C010C00u;
    r.psel[2] = (r.neg & 4u) ? 0x0C050C04u : 0x0C010C00u;
    r.sp = 0;
    r.cur = 0u; // root node (always an inner node)
    r.leaf = TRAVERSAL_DONE;
}

// Tests the triangles of the postponed leaf (ANY: the first hit ends the traversal).
template <bool COUNT, bool ANY, bool SORTED>
__device__ __forceinline__ void leaf_test(const float4* __restrict__ tris, RayState& r, uint32_t ray_mask,
                                          TraversalCount& count) {
    const uint32_t first = (r.leaf & 0x7FFFFFFFu) >> 3;
    const uint32_t cnt = (r.leaf & 7u) + 1u;
    // two records per round, both fetched before either is tested (one memory round trip)
    for (uint32_t k = 0; k < cnt; k += 2) {
        const uint32_t a = first + k, b = first + min(k + 1u, cnt - 1u);
        const float4 A0 = tris[3 * a], B0 = tris[3 * a + 1], C0 = tris[3 * a + 2];
        const float4 A1 = tris[3 * b], B1 = tris[3 * b + 1], C1 = tris[3 * b + 2];
        test_triangle(A0, B0, C0, r.o, r.d, r.tmin, r.tmax, ray_mask, r.best);
        if (k + 1u < cnt) test_triangle(A1, B1, C1, r.o, r.d, r.tmin, r.tmax, ray_mask, r.best);
    }
    if constexpr (COUNT) count.tris += cnt;
    r.leaf = TRAVERSAL_DONE;
    r.klim = far_limit<SORTED>(r.tmax, r.best.t);
    if constexpr (ANY) {
        if (r.best.id != TRAVERSAL_DONE) {
            r.cur = TRAVERSAL_DONE;
            r.sp = 0;
        }
    }
}

// Entry of a slot from its node's child base and triangle base and its code byte (bvh.h).
__device__ __forceinline__ uint32_t code_entry(uint32_t child_base, uint32_t tri_base, uint32_t code) {
    return (code >= BVH8_INNER ? child_base - uint32_t(BVH8_INNER) : LEAF_FLAG | (tri_base << 3)) + code;
}

// Grouped BVH8 stack entries: a node index (< 2^24) and, in the top byte, the node's hit
// children not yet visited as a mask over visiting positions (position i = slot i ^ r.neg).
constexpr uint32_t BVH8_GROUP_NODE = 0xFFFFFFu;

// The trees as the traversal reads them. W: children per node.
struct DeviceBVH4 { // near-first order by sorted distances, one stack entry per pushed child
    static constexpr int W = 4;
    static constexpr bool SORTED = true;
    const BVH4Node* nodes;
    const float4* tris; // TriRecord as 3 x float4
};
struct DeviceBVH8 {
    static constexpr int W = 8;
    static constexpr bool SORTED = true;
    const BVH8Node* nodes;
    const float4* tris;
};
struct DeviceBVH8G { // octant visiting order, one stack group per node
    static constexpr int W = 8;
    static constexpr bool SORTED = false;
    const BVH8Node* nodes;
    const float4* tris;
};

// Next entry to visit: sorted trees pop a ready entry; grouped BVH8 takes the first remaining child
// of the top group (re-reading its node's 16-byte header) and drops the group once it is empty.
template <class BVH> __device__ __forceinline__ uint32_t pop_next(const BVH bvh, RayState& r, const LaneStack& stk) {
    if (r.sp == 0) return TRAVERSAL_DONE;
    if constexpr (BVH::SORTED) {
        return stack_peek(stk, --r.sp);
    } else {
        const uint32_t g = stack_peek(stk, r.sp - 1);
        const uint32_t node = g & BVH8_GROUP_NODE;
        const uint32_t m = g >> 24;
        const uint4 h1 = reinterpret_cast<const uint4*>(bvh.nodes + node)[1];
        const uint32_t rest = m & (m - 1u);
        if (rest == 0u) {
            r.sp--;
        } else {
            stack_poke(stk, r.sp - 1, node | (rest << 24));
        }
        const uint32_t c = uint32_t(__builtin_ctz(m)) ^ r.neg;
        return code_entry(h1.x, h1.y, __builtin_amdgcn_perm(h1.w, h1.z, c | 0x0C0C0C00u));
    }
}

// A node as read: grid origin and steps, bases, codes, and per axis the lo / hi plane bytes of
// children 0-3 and (W = 8) 4-7.
template <int W> struct NodeData {
    float px, py, pz;
    int ex, ey, ez;
    uint32_t child_base, tri_base, code[W / 4];
    uint32_t lo[3][W / 4], hi[3][W / 4];
};
// IN_ORDER keeps the five loads of a BVH8 node together and ascending, the wait after the last. Octant
// order, whose long incoherent traversals wait on the L1 and thrash it, wants that: 16.8 M incoherent
// rays in a million triangles take 30.2 ms (30.0 on another card) against 30.6 (30.4) in the order the
// compiler picks (48, 32, 16, 0, then 64). Sorted order is left to the compiler (the 1080p GBuffer pass:
// 404 us, 412 in order).
template <bool IN_ORDER> __device__ __forceinline__ void next_load() {
    if constexpr (IN_ORDER) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    }
}
template <bool IN_ORDER> __device__ __forceinline__ NodeData<8> load_node(const BVH8Node* n) {
    const uint4* p = reinterpret_cast<const uint4*>(n);
    const uint4 h0 = p[0];
    next_load<IN_ORDER>();
    const uint4 h1 = p[1];
    next_load<IN_ORDER>();
    const uint4 qx = p[2];
    next_load<IN_ORDER>();
    const uint4 qy = p[3];
    next_load<IN_ORDER>();
    const uint4 qz = p[4];
    next_load<IN_ORDER>();
    return NodeData<8>{__uint_as_float(h0.x), __uint_as_float(h0.y), __uint_as_float(h0.z),
                       int(int8_t(h0.w & 0xFFu)), int(int8_t((h0.w >> 8) & 0xFFu)), int(int8_t((h0.w >> 16) & 0xFFu)),
                       h1.x, h1.y, {h1.z, h1.w},
                       {{qx.x, qx.y}, {qy.x, qy.y}, {qz.x, qz.y}}, {{qx.z, qx.w}, {qy.z, qy.w}, {qz.z, qz.w}}};
}
template <bool> __device__ __forceinline__ NodeData<4> load_node(const BVH4Node* n) {
    const uint4* p = reinterpret_cast<const uint4*>(n);
    const uint4 h0 = p[0], h1 = p[1], h2 = p[2];
    return NodeData<4>{__uint_as_float(h0.x & BVH4_ORIGIN_MASK), __uint_as_float(h0.y & BVH4_ORIGIN_MASK),
                       __uint_as_float(h0.z & BVH4_ORIGIN_MASK), int(int8_t(h0.x & 0xFFu)), int(int8_t(h0.y & 0xFFu)),
                       int(int8_t(h0.z & 0xFFu)), h0.w, h1.x, {h1.y}, {{h1.z}, {h2.x}, {h2.z}}, {{h1.w}, {h2.y}, {h2.w}}};
}

// Slab tests of the node's W child boxes: entry and exit distance per child (tn clamped to the
// ray's near limit, tf not clamped to its far limit).
//
// Distances are taken in the node's grid: a plane at grid coordinate q lies at q 2^e + p, so its
// distance is q (2^e / d) + (p / d - o / d) = fma(q, a, b) with a = 2^e ix (exact: a power-of-two
// scale) and b = fma(p, ix, -ox) once per node and axis. A plane's byte, zero-extended to 16
// bits by the byte permute that picks near or far planes of two children at once, is the half
// float q 2^-24 (a denormal, exact), which the mixed-precision FMA takes as its first operand; a
// carries the factor 2^24. So a plane costs half a permute and an FMA, against half a permute of
// four, a byte conversion and an FMA before (the same values: q a is rounded once, in the FMA).
template <int W>
__device__ __forceinline__ void slab_tests(const NodeData<W>& n, const RayState& r, float (&tn)[W], float (&tf)[W]) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const float a[3] = {ldexpf(r.ix, n.ex + 24), ldexpf(r.iy, n.ey + 24), ldexpf(r.iz, n.ez + 24)};
    const float b[3] = {__builtin_fmaf(n.px, r.ix, -r.ox), __builtin_fmaf(n.py, r.iy, -r.oy),
                        __builtin_fmaf(n.pz, r.iz, -r.oz)};
#pragma unroll
    for (int p = 0; p < W / 2; p++) { // children 2 p, 2 p + 1
        const int w = p >> 1;
        float nr[3][2], fr[3][2];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const uint32_t sel = r.psel[k] + ((p & 1) ? 0x00020002u : 0u);
            const h2 qn = __builtin_bit_cast(h2, __builtin_amdgcn_perm(n.hi[k][w], n.lo[k][w], sel));
            const h2 qf = __builtin_bit_cast(h2, __builtin_amdgcn_perm(n.lo[k][w], n.hi[k][w], sel));
            nr[k][0] = __builtin_fmaf(float(qn.x), a[k], b[k]);
            nr[k][1] = __builtin_fmaf(float(qn.y), a[k], b[k]);
            fr[k][0] = __builtin_fmaf(float(qf.x), a[k], b[k]);
            fr[k][1] = __builtin_fmaf(float(qf.y), a[k], b[k]);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            tn[2 * p + j] = fmaxf(fmaxf(nr[0][j], nr[1][j]), fmaxf(nr[2][j], r.t0));
            tf[2 * p + j] = fminf(fminf(fr[0][j], fr[1][j]), fr[2][j]);
        }
    }
}

__device__ __forceinline__ int med3(int a, int b, int c) { return max(min(a, b), min(max(a, b), c)); }

// One inner-node step (r.cur is an inner node), near-first by sorted entry distance: sort the
// children near to far, push the hit ones but the nearest, continue with the nearest.
//
// The sort key of a child is its entry distance's bit pattern with the slot's code byte in place of
// the low byte (one byte permute; a missed box: KEY_MISS), so a key holds all that a pushed child's
// entry needs. The far limit is applied to the sorted keys (key <= klim), not to every box. Keys are
// sorted by insertion: a key d goes into a sorted list s by out[i] = med3(s[i - 1], s[i], d), one
// instruction per element (33 for eight keys, 7 for four, against 38 and 10 of a compare-exchange
// network).
// An empty slot (an inverted box) can only pass if all its plane distances round to one value; it
// then reads as a leaf of one record at most 30 past the node's own, which the triangle array's
// padding keeps in bounds: one more triangle tested, or a null record. So slots are not checked
// for being empty.
// Only the visiting order depends on the keys; which children are visited does not.
template <bool COUNT, class BVH>
__device__ __forceinline__ void node_step(const BVH bvh, RayState& r, const LaneStack& stk, TraversalCount& count) {
    constexpr int W = BVH::W;
    if constexpr (COUNT) count.nodes++;
    const NodeData<W> n = load_node<!BVH::SORTED>(bvh.nodes + r.cur);
    float tn[W], tf[W];
    slab_tests(n, r, tn, tf);
    if constexpr (BVH::SORTED) {
        int key[W];
#pragma unroll
        for (int c = 0; c < W; c++) {
            const uint32_t k = __builtin_amdgcn_perm(__float_as_uint(tn[c]), n.code[c >> 2], 0x07060500u | uint32_t(c & 3));
            const int d = tn[c] <= tf[c] ? int(k) : KEY_MISS;
            // key[0 .. c - 1] is sorted: insert d
            int prev = d;
#pragma unroll
            for (int i = 0; i < c; i++) {
                const int s = key[i];
                key[i] = i == 0 ? min(s, d) : med3(prev, s, d);
                prev = s;
            }
            key[c] = c == 0 ? d : max(prev, d);
        }
        const uint32_t inner_base = n.child_base - uint32_t(BVH8_INNER), leaf_base = LEAF_FLAG | (n.tri_base << 3);
        auto entry_of = [&](int k) {
            const uint32_t code = uint32_t(k) & 0xFFu;
            return (code >= BVH8_INNER ? inner_base : leaf_base) + code;
        };
        // far to near; the whole wave writes to LDS unless a lane's stack may leave it
        if (__any(r.sp > TRACE_LDS_STACK - (W - 1))) {
#pragma unroll
            for (int c = W - 1; c >= 1; c--)
                if (key[c] <= r.klim) stack_push(stk, r.sp, entry_of(key[c]));
        } else {
#pragma unroll
            for (int c = W - 1; c >= 1; c--)
                if (key[c] <= r.klim) ((lds_u32)stk.lds)[r.sp++ * TRACE_BLOCK] = entry_of(key[c]);
        }
        r.cur = key[0] <= r.klim ? entry_of(key[0]) : pop_next(bvh, r, stk);
    } else {
        // Octant order: continue with the first hit child in the ray's visiting order and push the
        // others as one group. Fewer instructions per node than the sorted step, but a pop re-reads
        // a node header: it wins on long incoherent traversals and loses where pops are frequent.
        // The builder puts a child in the slot of the node corner it lies toward (bit a: high end of
        // axis a), so a ray whose direction signs are r.neg meets them roughly in the order
        // slot = i ^ r.neg, i = 0..7 (the ordering of compressed wide BVHs, Ylitie, Karras and
        // Laine 2017); the hit mask is permuted into that order by three conditional bit-group
        // swaps, and no distances are sorted.
        const float tlim = __uint_as_float(uint32_t(r.klim));
        uint32_t hm = 0u; // bit c: slot c is hit
#pragma unroll
        for (int c = 0; c < 8; c++) hm |= tn[c] <= fminf(tf[c], tlim) ? (1u << c) : 0u;
        // position i of the visiting order is slot i ^ neg: swap bit pairs, pairs of pairs, nibbles
        uint32_t pm = hm;
        if (r.neg & 1u) pm = ((pm & 0x55u) << 1) | ((pm >> 1) & 0x55u);
        if (r.neg & 2u) pm = ((pm & 0x33u) << 2) | ((pm >> 2) & 0x33u);
        if (r.neg & 4u) pm = ((pm & 0x0Fu) << 4) | (pm >> 4);
        if (pm == 0u) {
            r.cur = pop_next(bvh, r, stk);
            return;
        }
        const uint32_t rest = pm & (pm - 1u);
        if (rest != 0u) stack_push(stk, r.sp, r.cur | (rest << 24));
        const uint32_t c = uint32_t(__builtin_ctz(pm)) ^ r.neg;
        r.cur = code_entry(n.child_base, n.tri_base, __builtin_amdgcn_perm(n.code[1], n.code[0], c | 0x0C0C0C00u));
    }
}

// Moves a leaf entry in `cur` into the (empty) postponed slot and takes the next entry, so the
// lane can keep stepping through inner nodes while its leaf waits for the wave's next leaf
// phase (speculative traversal, Aila & Laine 2009).
template <class BVH>
__device__ __forceinline__ void postpone_leaf(const BVH& bvh, RayState& r, const LaneStack& stk) {
    if (r.leaf == TRAVERSAL_DONE && is_leaf(r.cur)) {
        r.leaf = r.cur;
        r.cur = pop_next(bvh, r, stk);
    }
}

// What the lanes of a wave keep in LDS beside their stacks. Slot k belongs to the ray that lane k
// loaded last; it is used once lanes share rays (trace_persistent).
struct WaveShared {
    unsigned long long key[64]; // closest hit of the ray so far: ordered t, then id (hit_key)
    float t[64], u[64], v[64];  // that hit
    uint32_t workers[64];       // lanes working on the ray
    uint32_t giver[64];         // k-th lane that gives a stack entry away
};

// Idle lanes of a wave without fresh rays before they take work from the others (4, 16 and 32 measured
// within 1 % of each other).
constexpr uint32_t SHARE_IDLE = 16;

// (t, id) as one integer that orders hits as the traversal does: smaller t first (-0 is 0), ties to
// the lower id; a miss (t = inf, id = ~0) last.
__device__ __forceinline__ unsigned long long hit_key(const HitRec& h) {
    const uint32_t b = __float_as_uint(h.t + 0.0f);
    return (static_cast<unsigned long long>(b ^ ((b >> 31) ? 0xFFFFFFFFu : 0x80000000u)) << 32) | h.id;
}

// LDS traffic between the lanes of one wave: the hardware keeps it in order; this keeps the compiler
// from moving accesses across.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Rank of a lane among the lanes of a set.
__device__ __forceinline__ uint32_t lane_rank(uint64_t mask, uint32_t lane) {
    return uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
}

// After a leaf test in a shared wave: the lane's hit goes to its ray's slot if it is the closest so
// far, and the ray's closest hit comes back as the limit of the lane's further tests.
// found: the test found the lane's hit (its u and v are then the lane's own).
template <bool ANY, bool SORTED>
__device__ __forceinline__ void share_hit(WaveShared& ws, RayState& r, uint32_t slot, bool found) {
    const unsigned long long key = hit_key(r.best);
    if (found) atomicMin(&ws.key[slot], key);
    wave_fence();
    const unsigned long long now = ws.key[slot];
    if (now == key) {
        if (found) {
            ws.t[slot] = r.best.t;
            ws.u[slot] = r.best.u;
            ws.v[slot] = r.best.v;
        }
    } else {
        // another lane's hit is closer: its (t, id) bounds this lane's tests (u and v stay in the slot)
        const uint32_t b = uint32_t(now >> 32);
        r.best.t = __uint_as_float(b ^ ((b >> 31) ? 0x80000000u : 0xFFFFFFFFu));
        r.best.id = uint32_t(now);
        r.klim = far_limit<SORTED>(r.tmax, r.best.t);
    }
    if constexpr (ANY) {
        if (r.best.id != TRAVERSAL_DONE) {
            r.cur = TRAVERSAL_DONE;
            r.sp = 0;
        }
    }
}

// Persistent closest-hit loop of one wave: every lane runs one traversal step per iteration and,
// when its ray is done, hands the hit to `sink` and later takes a fresh ray from `src`, so lanes
// with short rays do not idle while others finish long ones.
//
// Ray indices are handed out in wave-private chunks, so the cursor `work` (zero at launch) sees a few
// atomics per wave instead of one per refill (it takes 75 to 120 M a second): every wave first owns a
// static chunk of n / (2 * waves) rays (rounded down to whole waves of 64), then claims guided chunks
// of (unclaimed rays) / (2 * waves), 64..1024 rays, from `work`. A SHARE launch has so few rays per
// wave that the claims would be its longest part: seven eighths of its rays are owned, in batches of
// 64 that go round the waves (neighbouring camera rays cost alike: a contiguous range per wave makes
// the 1080p GBuffer pass 566 us instead of 440), and with at most 64 rays per wave all are, evenly.
//
// Src::CURSORS: the rays are halved as without SHARE, with a cursor per 1/8 of them (ray_claims.h).
//
// Refilled lanes issue their ray loads before the still-active lanes' traversal step, so both
// wait on one memory round trip.
//
// Sharing (SHARE): once a wave has no fresh rays left, idle lanes take stack entries from lanes that
// still have some and work on those rays too, so the end of a launch, and all of a small one, is
// as long as its longest ray's work spread over the wave and not as its longest ray. A lane's ray
// is then named by a slot; leaf tests merge hits there (share_hit), and the last lane to finish work
// on a ray stores its hit. The result is the same: the closest (t, id) over all leaves reached.
// A wave whose refill threshold is 64 (it loads a batch when all its lanes are idle) shares every
// batch (a 512x512 frame so tuned 796 -> 682 us).
template <bool COUNT, bool ANY, bool SHARE, class Src, class Sink, class BVH>
__device__ __forceinline__ void trace_persistent(const BVH bvh, const Src& src, const Sink& sink, uint32_t n,
                                                 uint32_t* work, uint32_t ray_mask, const LaneStack& stk, WaveShared& ws,
                                                 TraversalCount& count, uint32_t refill, uint32_t leaf_lanes, float dir_min) {
    const uint32_t lane = __lane_id();
    const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    RayClaims claims = one_cursor(n, wave, waves);
    uint32_t pool, pool_end, dyn0; // positions of the share (claim_ray); dynamic claims start at dyn0
    uint32_t batches = 0, batch = 0; // SHARE: batches of 64 rays this wave owns, taken so far
    if (SHARE && !Src::CURSORS && n <= 64u * uint64_t(waves)) {
        const uint32_t each = (n + waves - 1u) / waves;
        pool = uint32_t(min(uint64_t(wave) * each, uint64_t(n)));
        pool_end = min(pool + each, n);
        dyn0 = n;
    } else if (SHARE && !Src::CURSORS) {
        batches = uint32_t(uint64_t(n) * 7u / (uint64_t(waves) * (8u * 64u)));
        dyn0 = batches * waves * 64u;
        pool = pool_end = 0u;
    } else {
        if constexpr (Src::CURSORS) {
            claims = many_cursors(n, blockIdx.x, gridDim.x, threadIdx.x >> 6, blockDim.x >> 6);
            work += claims.home * CURSOR_STRIDE;
            n = claims.n;
        }
        const uint32_t c0 = (n / (2u * claims.waves)) & ~63u;
        dyn0 = c0 * claims.waves; // <= n / 2
        pool = claims.wave * c0;
        pool_end = pool + c0;
    }
    uint32_t seen = dyn0;
    bool claims_done = dyn0 >= n;
    RayState r;
    r.cur = TRAVERSAL_DONE;
    r.sp = 0;
    bool active = false;
    bool sharing = false; // wave-uniform
    uint32_t slot = lane;
    uint32_t idx = 0;
    while (true) {
        const uint64_t idle = __ballot(!active);
        const uint32_t nidle = uint32_t(__popcll(idle));
        bool fresh = false;
        const bool more = !(claims_done && pool == pool_end) || (SHARE && batch < batches); // fresh rays for this wave
        if (!(nidle >= refill && more)) {
            // a wave that refills only when all its lanes are idle (refill 64) shares every batch
            if (SHARE && (!more || refill >= 64u)) {
                const bool can_give = active && r.sp > 0 && r.sp <= TRACE_LDS_STACK;
                const uint64_t givers = __ballot(can_give);
                if (nidle >= SHARE_IDLE && givers != 0) {
                    if (!sharing) {
                        sharing = true;
                        if (active) {
                            ws.key[lane] = hit_key(r.best);
                            ws.t[lane] = r.best.t;
                            ws.u[lane] = r.best.u;
                            ws.v[lane] = r.best.v;
                            ws.workers[lane] = 1u;
                        }
                    }
                    const uint32_t pairs = min(nidle, uint32_t(__popcll(givers)));
                    const uint32_t rank = lane_rank(can_give ? givers : idle, lane);
                    const bool give = can_give && rank < pairs, take = !active && rank < pairs;
                    if (give) ws.giver[rank] = lane;
                    wave_fence();
                    const uint32_t from = take ? ws.giver[rank] : lane;
                    const f3 o{__shfl(r.o.x, int(from)), __shfl(r.o.y, int(from)), __shfl(r.o.z, int(from))};
                    const f3 d{__shfl(r.d.x, int(from)), __shfl(r.d.y, int(from)), __shfl(r.d.z, int(from))};
                    const float tmin = __shfl(r.tmin, int(from)), tmax = __shfl(r.tmax, int(from));
                    const float bt = __shfl(r.best.t, int(from));
                    const uint32_t bid = __shfl(r.best.id, int(from));
                    const uint32_t gslot = __shfl(slot, int(from)), gidx = __shfl(idx, int(from));
                    const int gsp = __shfl(r.sp, int(from));
                    if (take) {
                        // the giver's next entry, the nearest of its pending ones
                        const uint32_t e = ((lds_u32)(stk.lds + (int(from) - int(lane))))[(gsp - 1) * TRACE_BLOCK];
                        ray_begin<BVH::SORTED>(r, o, d, tmin, tmax, dir_min);
                        r.best.t = bt;
                        r.best.id = bid;
                        r.klim = far_limit<BVH::SORTED>(tmax, bt);
                        slot = gslot;
                        idx = gidx;
                        atomicAdd(&ws.workers[slot], 1u);
                        active = true;
                        if constexpr (BVH::SORTED) {
                            r.cur = e;
                        } else { // a group of children
                            stack_push(stk, r.sp, e);
                            r.cur = pop_next(bvh, r, stk);
                        }
                        postpone_leaf(bvh, r, stk);
                    }
                    if (give) r.sp--;
                }
            }
        } else {
            sharing = sharing && nidle < 64u; // all lanes idle: no slot is in use
            const uint32_t avail = pool_end - pool;
            uint32_t lo = 0, hi = 0;
            if (SHARE && avail < nidle && batch < batches) {
                lo = (batch * waves + wave) * 64u;
                hi = lo + 64u;
                batch++;
            } else if (avail < nidle && !claims_done) {
                const uint32_t left = n - (seen < n ? seen : n);
                const uint32_t chunk = min(max((left / (2u * claims.waves)) & ~63u, 64u), 1024u);
                const uint32_t leader = uint32_t(__ffsll((unsigned long long)idle) - 1);
                uint32_t got = 0;
                if (lane == leader) got = atomicAdd(work, chunk);
                const uint64_t base = uint64_t(__shfl(got, int(leader))) + dyn0;
                seen = base < n ? uint32_t(base) : n;
                if (base < n) {
                    lo = uint32_t(base);
                    hi = uint32_t(base + chunk < n ? base + chunk : n);
                }
                if (base + chunk >= n) claims_done = true;
            }
            if (!active) {
                const uint32_t k = lane_rank(idle, lane);
                uint32_t my = TRAVERSAL_DONE;
                if (k < avail) {
                    my = pool + k;
                } else if (k - avail < hi - lo) {
                    my = lo + (k - avail);
                }
                if (my != TRAVERSAL_DONE) {
                    idx = Src::CURSORS ? claim_ray(claims, my) : my;
                    slot = lane;
                    src.load(idx, r.o, r.d, r.tmin, r.tmax); // this lane's state is dead until ray_begin
                    fresh = true;
                }
            }
            if (avail >= nidle) {
                pool += nidle;
            } else {
                pool = lo + min(nidle - avail, hi - lo);
                pool_end = hi;
            }
        }
        // One wave-uniform phase per iteration: an inner-node step for every lane whose current
        // entry is an inner node, or a leaf test for every lane with a postponed leaf. Leaf
        // phases run once `leaf_lanes` lanes can do nothing but their leaf (or no lane has an
        // inner node left), so both code paths run with most lanes active.
        const bool inner_ok = active && is_inner(r.cur);
        const bool has_leaf = active && r.leaf != TRAVERSAL_DONE;
        const uint64_t mi = __ballot(inner_ok);
        const uint64_t ml = __ballot(has_leaf);
        if ((mi | ml) == 0 && __ballot(fresh) == 0) break;
        const bool leaf_phase = mi == 0 || uint32_t(__popcll(ml & ~mi)) >= leaf_lanes;
        if (leaf_phase) {
            if (has_leaf) {
                const uint32_t before = r.best.id;
                leaf_test<COUNT, ANY, BVH::SORTED>(bvh.tris, r, ray_mask, count);
                if (SHARE && sharing) share_hit<ANY, BVH::SORTED>(ws, r, slot, r.best.id != before);
            }
        } else {
            if (inner_ok) node_step<COUNT>(bvh, r, stk, count);
        }
        if (active) {
            postpone_leaf(bvh, r, stk);
            if (r.cur == TRAVERSAL_DONE && r.leaf == TRAVERSAL_DONE) {
                if (SHARE && sharing) {
                    wave_fence();
                    if (atomicSub(&ws.workers[slot], 1u) == 1u) {
                        r.best = HitRec{uint32_t(ws.key[slot]), ws.t[slot], ws.u[slot], ws.v[slot]};
                        sink.store(idx, r.best);
                    }
                } else {
                    sink.store(idx, r.best);
                }
                active = false;
            }
        }
        if (fresh) {
            ray_begin<BVH::SORTED>(r, r.o, r.d, r.tmin, r.tmax, dir_min);
            active = true;
        }
    }
}

} // namespace mrt

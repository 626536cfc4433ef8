// 4- and 8-wide quantised BVHs for the gfx950 traversal kernels: layouts and host builder.
//
// Replaces the driver acceleration-structure build of the reference
// (src/merian/vk/raytrace/as_builder_blas.cpp:137, as_builder_tlas.cpp:131). Hit results do not
// depend on the tree shape: traversal is conservative and ties at equal t go to the lowest
// triangle id, so any correct tree returns the brute-force closest hit.
#pragma once

#include <stdint.h>

#include <vector>

namespace mrt {

// Triangle record in leaf order: the Moller-Trumbore operands, three 16-byte loads.
//   a = (v0.xyz, id bits)   b = (e1.xyz, flags bits)   c = (e2.xyz, 0)
// flags: bit 0 = back-face culling on, bits 8..15 = 8-bit instance mask.
struct alignas(16) TriRecord {
    float a[4], b[4], c[4];
};

// Leaf stack entries: bit 31 set, first record in bits 3..30, (count - 1) in bits 0..2.
constexpr uint32_t LEAF_FLAG = 0x80000000u;
constexpr int MAX_LEAF = 8; // most triangles per leaf the encoding allows (the build default is 4)

// 8-wide node with child boxes quantised to 8 bits on a per-node power-of-two grid (80 bytes,
// five 16-byte loads): child box = fma(q, 2^e, origin) per plane, rounded outward, so that every
// decoded box contains the padded child box. Inner children are stored consecutively from child_base
// in slot order; the triangles of the leaf children consecutively from tri_base.
// One code byte per slot makes the slot's traversal entry a select and an add:
//   leaf:  (first triangle - tri_base) << 3 | (count - 1)   (<= BVH8_LEAF_CODE_MAX)
//   empty: BVH8_EMPTY
//   inner: BVH8_INNER + rank among the inner children
// so entry = (inner ? child_base - BVH8_INNER : LEAF | tri_base << 3) + code.
constexpr uint8_t BVH8_EMPTY = 0xF0, BVH8_INNER = 0xF8;
constexpr int BVH8_MAX_LEAF = 4; // 7 leaves of 4 before a slot: offset 28, code 227
constexpr uint32_t BVH8_LEAF_CODE_MAX = 28u << 3 | 3u;
struct alignas(16) BVH8Node {
    float px, py, pz;       // grid origin
    int8_t ex, ey, ez;      // grid step 2^e per axis
    uint8_t inner_mask;     // bit k: slot k is an inner child
    uint32_t child_base;    // node index of the first inner child
    uint32_t tri_base;      // first triangle record of the leaf children
    uint8_t code[8];        // per slot, as above
    uint8_t qlox[8], qhix[8], qloy[8], qhiy[8], qloz[8], qhiz[8]; // empty slot: lo 255, hi 0
};
static_assert(sizeof(BVH8Node) == 80, "BVH8Node must be 80 bytes");
static_assert(BVH8_LEAF_CODE_MAX < BVH8_EMPTY, "leaf codes below the sentinels");

// The same node for four children, 48 bytes: three 16-byte loads per visit (a traversal's loads are
// scattered, one L1 access per lane and load, and the L1's address path is as busy as the vector
// units: full-precision boxes cost seven loads). The grid exponent of an axis is the low byte of its
// origin, whose float keeps 24 bits (rounded down).
constexpr uint32_t BVH4_ORIGIN_MASK = 0xFFFFFF00u;
struct alignas(16) BVH4Node {
    uint32_t px, py, pz;    // grid origin (high 24 bits of the float) | exponent (int8) per axis
    uint32_t child_base;
    uint32_t tri_base;
    uint8_t code[4];        // as BVH8Node.code
    uint8_t qlox[4], qhix[4], qloy[4], qhiy[4], qloz[4], qhiz[4]; // empty slot: lo 255, hi 0
};
static_assert(sizeof(BVH4Node) == 48, "BVH4Node must be 48 bytes");
static_assert(((3 * MAX_LEAF) << 3 | (MAX_LEAF - 1)) < BVH8_EMPTY, "leaf codes below the sentinels");

// Null triangle records a device copy of `tris` ends with: the traversal may read an empty slot as a
// leaf of one record, (BVH8_EMPTY >> 3) past a node's tri_base (mrt_trace.h).
constexpr uint32_t TRI_PADDING = (BVH8_EMPTY >> 3) + 1u;

struct BVH4 {
    std::vector<BVH4Node> nodes; // nodes[0] is the root
    std::vector<TriRecord> tris; // per node, its leaf children's triangles in slot order
    uint32_t depth = 0;          // longest root-to-leaf path in nodes
    int max_exp = -126;          // largest grid exponent
};

struct BVH8 {
    std::vector<BVH8Node> nodes; // nodes[0] is the root
    std::vector<TriRecord> tris; // per node, its leaf children's triangles in slot order
    uint32_t depth = 0;
    int max_exp = -126;
};

// Smallest magnitude a direction component d takes in the box tests: 1e-20, and so large that
// 2^(max_exp + 24) / d, the scale of the slab tests, stays finite (scenes beyond 2^45 units only).
inline float bvh_dir_min(int max_exp) {
    const int e = max_exp + 24 - 127;
    return e > -66 ? __builtin_ldexpf(1.0f, e < 126 ? e : 126) : 1e-20f;
}

// v0/e1/e2: per-triangle float[3] operands exactly as the intersection test uses them
// (e1 = v1 - v0, e2 = v2 - v0 rounded in float). flags as in TriRecord.
// max_leaf: most triangles per leaf (1..MAX_LEAF); traversal_cost: SAH cost of one node
// visit relative to one triangle test.
BVH8 build_bvh8(const float* v0, const float* e1, const float* e2, const uint32_t* flags, uint32_t n,
                int threads, int max_leaf = 4, float traversal_cost = 1.0f);

BVH4 build_bvh4(const float* v0, const float* e1, const float* e2, const uint32_t* flags, uint32_t n,
                int threads, int max_leaf = 4, float traversal_cost = 1.0f);

} // namespace mrt

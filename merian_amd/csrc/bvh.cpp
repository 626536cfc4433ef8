// Binned-SAH BVH2 build, collapsed into the quantised BVH4 and BVH8 layouts of bvh.h.
//
// The reference leaves BVH construction to the Vulkan driver (PreferFastTrace for static mesh
// groups, src/merian-shaders/scene/scene.cpp:1116-1123). This builder is the project's own:
// 32-bin SAH per axis over centroid bounds, leaves of at most max_leaf (<= MAX_LEAF) triangles, top levels
// built in parallel threads. Child boxes are rounded outward and padded so that the slab test
// (one FMA per plane) can never reject a box containing a hit the triangle test reports.
#include "bvh.h"

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <thread>

namespace mrt {
namespace {

struct AABB {
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
    float hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    void grow(const AABB& b) {
        for (int k = 0; k < 3; k++) {
            lo[k] = std::min(lo[k], b.lo[k]);
            hi[k] = std::max(hi[k], b.hi[k]);
        }
    }
    void grow(const float* p) {
        for (int k = 0; k < 3; k++) {
            lo[k] = std::min(lo[k], p[k]);
            hi[k] = std::max(hi[k], p[k]);
        }
    }
    float area() const {
        const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
        if (dx < 0.f) return 0.f;
        return 2.f * (dx * dy + dy * dz + dz * dx);
    }
};

struct Prim {
    AABB box;
    float c[3];
};

struct Node2 {
    AABB box;
    int32_t left = -1, right = -1;
    uint32_t first = 0, count = 0;
};

constexpr int BINS = 32;

struct Builder {
    const std::vector<Prim>& prims;
    std::vector<uint32_t> idx;
    std::vector<Node2> nodes;
    std::atomic<uint32_t> next{1};
    int par_depth;
    uint32_t max_leaf = 4;
    float traversal_cost = 1.0f;

    Builder(const std::vector<Prim>& p, std::vector<uint32_t> order, int threads)
        : prims(p), idx(std::move(order)), nodes(std::max<size_t>(1, 2 * idx.size())) {
        par_depth = 0;
        while ((1 << par_depth) < threads && par_depth < 6) par_depth++;
    }

    void make_leaf(Node2& n, uint32_t b, uint32_t e) {
        n.left = n.right = -1;
        n.first = b;
        n.count = e - b;
    }

    void build(uint32_t ni, uint32_t b, uint32_t e, int depth) {
        Node2& node = nodes[ni];
        AABB box, cbox;
        for (uint32_t i = b; i < e; i++) {
            box.grow(prims[idx[i]].box);
            cbox.grow(prims[idx[i]].c);
        }
        node.box = box;
        const uint32_t n = e - b;
        if (n <= 1) {
            make_leaf(node, b, e);
            return;
        }
        // binned SAH over centroid bounds
        float best_cost = FLT_MAX;
        int best_axis = -1, best_split = 0;
        for (int ax = 0; ax < 3; ax++) {
            const float ext = cbox.hi[ax] - cbox.lo[ax];
            if (!(ext > 0.f)) continue;
            const float scale = float(BINS) / ext;
            AABB bb[BINS];
            uint32_t cnt[BINS] = {};
            for (uint32_t i = b; i < e; i++) {
                const Prim& p = prims[idx[i]];
                int k = int((p.c[ax] - cbox.lo[ax]) * scale);
                k = std::min(std::max(k, 0), BINS - 1);
                cnt[k]++;
                bb[k].grow(p.box);
            }
            float right_area[BINS];
            uint32_t right_cnt[BINS];
            AABB acc;
            uint32_t c = 0;
            for (int k = BINS - 1; k > 0; k--) {
                acc.grow(bb[k]);
                c += cnt[k];
                right_area[k] = acc.area();
                right_cnt[k] = c;
            }
            AABB lacc;
            uint32_t lc = 0;
            for (int k = 1; k < BINS; k++) {
                lacc.grow(bb[k - 1]);
                lc += cnt[k - 1];
                if (lc == 0 || right_cnt[k] == 0) continue;
                const float cost = lacc.area() * float(lc) + right_area[k] * float(right_cnt[k]);
                if (cost < best_cost) {
                    best_cost = cost;
                    best_axis = ax;
                    best_split = k;
                }
            }
        }
        const float leaf_cost = box.area() * float(n);
        uint32_t mid;
        if (best_axis < 0) {
            if (n <= max_leaf) {
                make_leaf(node, b, e);
                return;
            }
            mid = b + n / 2; // coincident centroids: split by index
        } else {
            if (n <= max_leaf && best_cost + traversal_cost * box.area() >= leaf_cost) {
                make_leaf(node, b, e);
                return;
            }
            const float ext = cbox.hi[best_axis] - cbox.lo[best_axis];
            const float scale = float(BINS) / ext;
            const float lo = cbox.lo[best_axis];
            auto it = std::partition(idx.begin() + b, idx.begin() + e, [&](uint32_t pi) {
                int k = int((prims[pi].c[best_axis] - lo) * scale);
                k = std::min(std::max(k, 0), BINS - 1);
                return k < best_split;
            });
            mid = uint32_t(it - idx.begin());
            if (mid == b || mid == e) mid = b + n / 2;
        }
        const uint32_t l = next.fetch_add(2);
        const uint32_t r = l + 1;
        node.left = int32_t(l);
        node.right = int32_t(r);
        node.count = 0;
        if (depth < par_depth && n > 65536) {
            std::thread t([&, l, b, mid, depth] { build(l, b, mid, depth + 1); });
            build(r, mid, e, depth + 1);
            t.join();
        } else {
            build(l, b, mid, depth + 1);
            build(r, mid, e, depth + 1);
        }
    }
};

// pad a child box outward: rounding of the FMA slab test and of the triangle test
void padded(const AABB& b, float mag, float lo[3], float hi[3]) {
    float ext = 0.f;
    for (int k = 0; k < 3; k++) ext = std::max(ext, b.hi[k] - b.lo[k]);
    const float pad = ext * (1.0f / 1024.0f) + mag * (1.0f / 65536.0f) + 1e-30f;
    for (int k = 0; k < 3; k++) {
        lo[k] = b.lo[k] - pad;
        hi[k] = b.hi[k] + pad;
    }
}

float down(double v) {
    float f = float(v);
    if (double(f) > v) f = std::nextafter(f, -INFINITY);
    return f;
}
float up(double v) {
    float f = float(v);
    if (double(f) < v) f = std::nextafter(f, INFINITY);
    return f;
}

} // namespace

namespace {

// Primitive boxes (as the intersection test sees the vertices) and the binned-SAH BVH2.
struct Prepared {
    std::vector<Prim> prims;
    std::vector<uint32_t> order;
    float mag = 0.f;
};

Prepared prepare(const float* v0, const float* e1, const float* e2, uint32_t n) {
    Prepared pr;
    pr.prims.resize(n);
    pr.order.reserve(n);
    for (uint32_t i = 0; i < n; i++) {
        Prim& p = pr.prims[i];
        bool ok = true;
        for (int k = 0; k < 3; k++) {
            // vertices as the intersection test sees them: v0, v0 + e1, v0 + e2 (exact in double)
            const double a = v0[3 * i + k], b = a + double(e1[3 * i + k]), c = a + double(e2[3 * i + k]);
            if (!std::isfinite(a) || !std::isfinite(b) || !std::isfinite(c)) ok = false;
            p.box.lo[k] = down(std::min(a, std::min(b, c)));
            p.box.hi[k] = up(std::max(a, std::max(b, c)));
            p.c[k] = float((std::min(a, std::min(b, c)) + std::max(a, std::max(b, c))) * 0.5);
        }
        if (!ok) continue; // a non-finite triangle can never be hit
        for (int k = 0; k < 3; k++)
            pr.mag = std::max(pr.mag, std::max(std::fabs(p.box.lo[k]), std::fabs(p.box.hi[k])));
        pr.order.push_back(i);
    }
    return pr;
}

void set_record(TriRecord& t, uint32_t i, const float* v0, const float* e1, const float* e2, const uint32_t* flags) {
    for (int c = 0; c < 3; c++) {
        t.a[c] = v0[3 * i + c];
        t.b[c] = e1[3 * i + c];
        t.c[c] = e2[3 * i + c];
    }
    std::memcpy(&t.a[3], &i, 4);
    std::memcpy(&t.b[3], &flags[i], 4);
    t.c[3] = 0.f;
}

// Children of a BVH2 node for a k-wide node: repeatedly open the largest inner child.
int gather_children(const std::vector<Node2>& n2, int32_t ni, int width, int32_t* kids) {
    int nk = 0;
    kids[nk++] = n2[ni].left;
    kids[nk++] = n2[ni].right;
    while (nk < width) {
        int best = -1;
        float best_area = -1.f;
        for (int i = 0; i < nk; i++) {
            const Node2& c = n2[kids[i]];
            if (c.left >= 0 && c.box.area() > best_area) {
                best_area = c.box.area();
                best = i;
            }
        }
        if (best < 0) break;
        const Node2 c = n2[kids[best]];
        kids[best] = c.left;
        kids[nk++] = c.right;
    }
    return nk;
}

// 8-bit grid of one node: origin, exponent per axis, quantised child planes containing `lo`/`hi`.
struct Quant {
    float p[3];
    int e[3];
};

// Rounds a grid origin down to the 24 bits a BVH4 node keeps of it.
float origin24(float v) {
    uint32_t b;
    std::memcpy(&b, &v, 4);
    if ((b & 0x80000000u) && (b & ~BVH4_ORIGIN_MASK)) b += 0x100u;
    b &= BVH4_ORIGIN_MASK;
    std::memcpy(&v, &b, 4);
    return v;
}

// width: the children per node of the tree, whose nodes keep the origin in 24 (4) or 32 (8) bits.
Quant node_grid(const float (*lo)[3], const float (*hi)[3], int nk, int width) {
    Quant q;
    for (int a = 0; a < 3; a++) {
        float mn = FLT_MAX, mx = -FLT_MAX;
        for (int k = 0; k < nk; k++) {
            mn = std::min(mn, lo[k][a]);
            mx = std::max(mx, hi[k][a]);
        }
        if (width == 4) mn = origin24(mn);
        q.p[a] = mn;
        const double ext = double(mx) - double(mn);
        int e = -126;
        if (ext > 0) {
            if (std::frexp(ext / 250.0, &e) == 0.5) e--; // ceil(log2(ext / 250))
            while (std::ldexp(250.0, e) < ext) e++;
        }
        q.e[a] = std::max(-126, std::min(127, e));
    }
    return q;
}

// Largest plane at most v, smallest plane at least v. The corrections run (almost) never: the test in
// front keeps the compiler from unrolling and vectorising them into every call (the collapse of 2 M
// triangles by one thread takes 230 ms instead of 690 to BVH4 nodes, 620 instead of 1,330 to BVH8).
uint8_t quant_lo(float v, float p, float s) {
    double q = std::floor((double(v) - double(p)) / double(s));
    int qi = int(std::max(0.0, std::min(255.0, q)));
    if (std::fmaf(float(qi), s, p) > v)
        while (qi > 0 && std::fmaf(float(qi), s, p) > v) qi--;
    return uint8_t(qi);
}

uint8_t quant_hi(float v, float p, float s) {
    double q = std::ceil((double(v) - double(p)) / double(s));
    int qi = int(std::max(0.0, std::min(255.0, q)));
    if (std::fmaf(float(qi), s, p) < v)
        while (qi < 255 && std::fmaf(float(qi), s, p) < v) qi++;
    return uint8_t(qi);
}

template <class Tree> struct Collapser {
    using Node = typename decltype(Tree::nodes)::value_type;
    static constexpr int W = sizeof(Node::code);
    const std::vector<Node2>& n2;
    const std::vector<uint32_t>& idx;
    const float *v0, *e1, *e2;
    const uint32_t* flags;
    Tree& out;
    float mag;

    // Places the node's children in slots by corner: slot bit a set = the child lies toward the
    // high end of axis a (children scored by their centre's offset from the node centre,
    // relative to the node's extent, greedily best pair first). A ray whose direction signs are
    // the bits o (bit a: negative along a) then meets the children roughly in slot order i ^ o.
    void assign_slots(const int32_t* kids, int nk, int32_t* slot_kid) const {
        for (int s = 0; s < 8; s++) slot_kid[s] = -1;
        float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
        float ctr[8][3];
        for (int k = 0; k < nk; k++) {
            const AABB& b = n2[kids[k]].box;
            for (int a = 0; a < 3; a++) {
                ctr[k][a] = 0.5f * (b.lo[a] + b.hi[a]);
                mn[a] = std::min(mn[a], b.lo[a]);
                mx[a] = std::max(mx[a], b.hi[a]);
            }
        }
        float score[8][8];
        for (int k = 0; k < nk; k++)
            for (int s = 0; s < 8; s++) {
                float sc = 0.f;
                for (int a = 0; a < 3; a++) {
                    const float ext = mx[a] - mn[a];
                    const float off = ext > 0.f ? (ctr[k][a] - 0.5f * (mn[a] + mx[a])) / ext : 0.f;
                    sc += ((s >> a) & 1) ? off : -off;
                }
                score[k][s] = sc;
            }
        bool kid_done[8] = {}, slot_done[8] = {};
        for (int n = 0; n < nk; n++) {
            int bk = -1, bs = -1;
            float best = -FLT_MAX;
            for (int k = 0; k < nk; k++)
                for (int s = 0; s < 8; s++)
                    if (!kid_done[k] && !slot_done[s] && score[k][s] > best) {
                        best = score[k][s];
                        bk = k;
                        bs = s;
                    }
            kid_done[bk] = slot_done[bs] = true;
            slot_kid[bs] = kids[bk];
        }
    }

    static void set_grid(BVH8Node& n, const Quant& g) {
        n.px = g.p[0];
        n.py = g.p[1];
        n.pz = g.p[2];
        n.ex = int8_t(g.e[0]);
        n.ey = int8_t(g.e[1]);
        n.ez = int8_t(g.e[2]);
    }
    static void set_grid(BVH4Node& n, const Quant& g) {
        uint32_t* p[3] = {&n.px, &n.py, &n.pz};
        for (int a = 0; a < 3; a++) {
            std::memcpy(p[a], &g.p[a], 4);
            *p[a] |= uint32_t(uint8_t(int8_t(g.e[a])));
        }
    }

    // fills out.nodes[me] from BVH2 node ni (or a lone leaf when ni is a leaf)
    void emit(int32_t ni, uint32_t me, uint32_t depth) {
        out.depth = std::max(out.depth, depth);
        int32_t kids[W];
        int nk;
        if (n2[ni].left < 0) {
            kids[0] = ni;
            nk = 1;
        } else {
            nk = gather_children(n2, ni, W, kids);
        }
        int32_t sk[W];
        if constexpr (W == 8) {
            assign_slots(kids, nk, sk);
        } else {
            for (int s = 0; s < W; s++) sk[s] = s < nk ? kids[s] : -1;
        }
        float lo[W][3], hi[W][3];
        for (int s = 0, k = 0; s < W; s++)
            if (sk[s] >= 0) {
                padded(n2[sk[s]].box, mag, lo[k], hi[k]);
                k++;
            }
        const Quant g = node_grid(lo, hi, nk, W);
        Node node;
        std::memset(&node, 0, sizeof(node));
        set_grid(node, g);
        out.max_exp = std::max(out.max_exp, std::max(g.e[0], std::max(g.e[1], g.e[2])));
        uint8_t* qlo[3] = {node.qlox, node.qloy, node.qloz};
        uint8_t* qhi[3] = {node.qhix, node.qhiy, node.qhiz};
        for (int k = 0; k < W; k++)
            for (int a = 0; a < 3; a++) {
                qlo[a][k] = 255;
                qhi[a][k] = 0;
            }
        int n_inner = 0;
        for (int k = 0; k < nk; k++)
            if (n2[kids[k]].left >= 0) n_inner++;
        node.child_base = uint32_t(out.nodes.size());
        out.nodes.resize(out.nodes.size() + size_t(n_inner));
        node.tri_base = uint32_t(out.tris.size());
        std::memset(node.code, BVH8_EMPTY, W);
        const float step[3] = {std::ldexp(1.0f, g.e[0]), std::ldexp(1.0f, g.e[1]), std::ldexp(1.0f, g.e[2])};
        uint32_t rank = 0;
        for (int s = 0, k = 0; s < W; s++) {
            if (sk[s] < 0) continue;
            const Node2& c = n2[sk[s]];
            for (int a = 0; a < 3; a++) {
                qlo[a][s] = quant_lo(lo[k][a], g.p[a], step[a]);
                qhi[a][s] = quant_hi(hi[k][a], g.p[a], step[a]);
            }
            k++;
            if (c.left >= 0) {
                if constexpr (W == 8) node.inner_mask |= uint8_t(1u << s);
                node.code[s] = uint8_t(BVH8_INNER + rank++);
            } else {
                const uint32_t off = uint32_t(out.tris.size()) - node.tri_base;
                node.code[s] = uint8_t(off << 3 | (c.count - 1u)); // count in [1, MAX_LEAF] ([1, BVH8_MAX_LEAF])
                for (uint32_t t = 0; t < c.count; t++) {
                    out.tris.emplace_back();
                    set_record(out.tris.back(), idx[c.first + t], v0, e1, e2, flags);
                }
            }
        }
        out.nodes[me] = node;
        uint32_t slot = node.child_base;
        for (int s = 0; s < W; s++)
            if (sk[s] >= 0 && n2[sk[s]].left >= 0) emit(sk[s], slot++, depth + 1);
    }
};

// Binned-SAH tree over the finite triangles, collapsed into `Tree`.
template <class Tree>
Tree build_tree(const float* v0, const float* e1, const float* e2, const uint32_t* flags, uint32_t n, int threads,
                int max_leaf, float traversal_cost) {
    using Node = typename decltype(Tree::nodes)::value_type;
    if (threads <= 0) threads = int(std::max(1u, std::thread::hardware_concurrency()));
    Prepared pr = prepare(v0, e1, e2, n);
    const float mag = pr.mag;
    const uint32_t m = uint32_t(pr.order.size());
    Builder bld(pr.prims, std::move(pr.order), threads);
    bld.max_leaf = uint32_t(std::max(max_leaf, 1));
    bld.traversal_cost = traversal_cost > 0.f ? traversal_cost : 1.0f;
    Tree out;
    out.nodes.emplace_back();
    if (m == 0) { // one node whose slots are all empty
        Node& node = out.nodes[0];
        std::memset(&node, 0, sizeof(node));
        std::memset(node.code, BVH8_EMPTY, sizeof(node.code));
        for (uint8_t* q : {node.qlox, node.qloy, node.qloz}) std::memset(q, 255, sizeof(node.code));
        out.depth = 1;
        out.max_exp = 0;
        return out;
    }
    bld.build(0, 0, m, 0);
    out.nodes.reserve(bld.next.load() / 2 + 2);
    out.tris.reserve(m);
    Collapser<Tree> col{bld.nodes, bld.idx, v0, e1, e2, flags, out, mag};
    col.emit(0, 0, 1);
    return out;
}

} // namespace

BVH4 build_bvh4(const float* v0, const float* e1, const float* e2, const uint32_t* flags, uint32_t n,
                int threads, int max_leaf, float traversal_cost) {
    return build_tree<BVH4>(v0, e1, e2, flags, n, threads, std::min(max_leaf, MAX_LEAF), traversal_cost);
}

BVH8 build_bvh8(const float* v0, const float* e1, const float* e2, const uint32_t* flags, uint32_t n,
                int threads, int max_leaf, float traversal_cost) {
    return build_tree<BVH8>(v0, e1, e2, flags, n, threads, std::min(max_leaf, BVH8_MAX_LEAF), traversal_cost);
}

} // namespace mrt

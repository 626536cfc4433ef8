// CPU check of the 4-wide quantised BVH (merian_amd/csrc/bvh.cpp): every child box, decoded as the
// kernel does (24-bit origin, exponent in its low byte), contains every triangle below it, every
// triangle appears exactly once, and the slot code bytes give the consecutive inner children and the
// leaf triangles in slot order. Positions cover negative and large origins, whose 24 bits are
// rounded down.
#include "../../merian_amd/csrc/bvh.h"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

using namespace mrt;

static int failures = 0;
#define CHECK(c)                                                       \
    do {                                                               \
        if (!(c)) {                                                    \
            if (failures < 10) std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #c); \
            failures++;                                                \
        }                                                              \
    } while (0)

static float decode(uint8_t q, uint32_t word) {
    const uint32_t o = word & BVH4_ORIGIN_MASK;
    float p;
    std::memcpy(&p, &o, 4);
    return std::fmaf(float(q), std::ldexp(1.0f, int(int8_t(word & 0xFFu))), p);
}

struct Box {
    float lo[3], hi[3];
};

// Visits node ni and all below it; counts the triangles in `seen`.
static void walk(const BVH4& b, uint32_t ni, std::vector<int>& seen, uint32_t depth) {
    CHECK(ni < b.nodes.size() && depth <= b.depth);
    if (ni >= b.nodes.size()) return;
    const BVH4Node& n = b.nodes[ni];
    const uint32_t p[3] = {n.px, n.py, n.pz};
    const uint8_t* qlo[3] = {n.qlox, n.qloy, n.qloz};
    const uint8_t* qhi[3] = {n.qhix, n.qhiy, n.qhiz};
    uint32_t inner = 0, tri = n.tri_base;
    for (int k = 0; k < 4; k++) {
        Box x;
        for (int a = 0; a < 3; a++) {
            x.lo[a] = decode(qlo[a][k], p[a]);
            x.hi[a] = decode(qhi[a][k], p[a]);
            CHECK(int(int8_t(p[a] & 0xFFu)) <= b.max_exp);
        }
        if (n.code[k] == BVH8_EMPTY) {
            for (int a = 0; a < 3; a++) CHECK(qlo[a][k] == 255 && qhi[a][k] == 0);
        } else if (n.code[k] >= BVH8_INNER) {
            CHECK(uint32_t(n.code[k] - BVH8_INNER) == inner);
            walk(b, n.child_base + inner++, seen, depth + 1);
        } else {
            const uint32_t cnt = (n.code[k] & 7u) + 1u;
            CHECK((uint32_t(n.code[k]) >> 3) == tri - n.tri_base && cnt <= uint32_t(MAX_LEAF));
            CHECK(size_t(tri) + cnt <= b.tris.size());
            if (size_t(tri) + cnt > b.tris.size()) return;
            for (uint32_t t = 0; t < cnt; t++, tri++) {
                const TriRecord& r = b.tris[tri];
                uint32_t id;
                std::memcpy(&id, &r.a[3], 4);
                CHECK(id < seen.size());
                if (id < seen.size()) seen[id]++;
                for (int a = 0; a < 3; a++) {
                    const float x0 = r.a[a], x1 = r.a[a] + r.b[a], x2 = r.a[a] + r.c[a];
                    CHECK(x.lo[a] <= std::fmin(x0, std::fmin(x1, x2)) && x.hi[a] >= std::fmax(x0, std::fmax(x1, x2)));
                }
            }
        }
    }
}

int main() {
    std::mt19937 rng(7);
    std::uniform_real_distribution<float> U(0.f, 1.f);
    struct Trial {
        uint32_t n;
        float scale, shift;
    };
    for (const Trial& tr : {Trial{1, 1, 0}, Trial{7, 1, -1}, Trial{1000, 1, -0.5f}, Trial{5000, 1e-3f, -700.f},
                            Trial{5000, 1e6f, -3e6f}, Trial{60000, 1000, -400.f}}) {
        std::vector<float> v0, e1, e2;
        std::vector<uint32_t> flags;
        for (uint32_t i = 0; i < tr.n; i++) {
            for (int k = 0; k < 3; k++) {
                v0.push_back(U(rng) * tr.scale + tr.shift);
                e1.push_back(0.02f * tr.scale * (U(rng) - 0.5f));
                e2.push_back(0.02f * tr.scale * (U(rng) - 0.5f));
            }
            flags.push_back(0xFF00u);
        }
        for (int leaf : {1, 2, 4, 8}) {
            const BVH4 b = build_bvh4(v0.data(), e1.data(), e2.data(), flags.data(), tr.n, 2, leaf, 1.0f);
            std::vector<int> seen(tr.n, 0);
            walk(b, 0, seen, 1);
            for (uint32_t i = 0; i < tr.n; i++) CHECK(seen[i] == 1);
            CHECK(b.tris.size() == tr.n);
        }
    }
    const BVH4 empty = build_bvh4(nullptr, nullptr, nullptr, nullptr, 0, 1, 4, 1.0f);
    CHECK(empty.nodes.size() == 1 && empty.tris.empty() && empty.depth == 1);
    std::vector<int> none;
    walk(empty, 0, none, 1);
    // the slab tests' scale 2^(e + 24) / d stays finite for every exponent, and ordinary scenes keep 1e-20
    CHECK(bvh_dir_min(10) == 1e-20f && bvh_dir_min(37) == 1e-20f);
    for (int e = -126; e <= 127; e++) CHECK(std::isfinite(std::ldexp(1.0f / bvh_dir_min(e), e < 102 ? e + 24 : 0)));
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("bvh4: all checks passed\n");
    return 0;
}

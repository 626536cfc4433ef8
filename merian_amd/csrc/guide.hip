// gfx950 kernels of the learned guide (include/merian_amd.h, MRT_MODE_GUIDED): hash-grid + SH
// encoding, the 64-wide MLP on MFMA (fp16 operands, fp32 accumulation), lobe packing for the
// shading kernel, and training (fused forward/backward per record tile, a weight-gradient GEMM
// over the batch, Adam). Layout conventions: mrt_guide.h.
#include "mrt_guide.h"

#include <rocprim/device/device_radix_sort.hpp>

namespace mrt {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// LDS traffic between the lanes of one wave: the hardware keeps it in order; this keeps the compiler
// from moving accesses across.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

constexpr int GB = 256;        // threads per block (4 waves)
constexpr int NT = 2;          // 16-query tiles per wave iteration
constexpr int WQ = 16 * NT;    // queries per wave iteration
constexpr int BQ = 4 * WQ;     // queries per block iteration
constexpr int IB = 512;        // threads per inference block (8 waves)
constexpr int IW = IB / 64;
constexpr int I_TILES = 4;     // inference: most 16-query tiles per wave iteration

__device__ __forceinline__ floatx4 mfma(const half8_t a, const half8_t b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Real spherical harmonics of degrees 0..3 (orthonormal on the sphere).
__device__ __forceinline__ float sh_coef(int k, float x, float y, float z) {
    switch (k) {
    case 0: return 0.28209479177387814f;
    case 1: return -0.48860251190291987f * y;
    case 2: return 0.48860251190291987f * z;
    case 3: return -0.48860251190291987f * x;
    case 4: return 1.0925484305920792f * (x * y);
    case 5: return -1.0925484305920792f * (y * z);
    case 6: return 0.94617469575755997f * (z * z) - 0.31539156525251999f;
    case 7: return -1.0925484305920792f * (x * z);
    case 8: return 0.54627421529603959f * (x * x - y * y);
    case 9: return 0.59004358992664352f * y * (-3.f * (x * x) + y * y);
    case 10: return 2.8906114426405538f * (x * y) * z;
    case 11: return 0.45704579946446572f * y * (1.f - 5.f * (z * z));
    case 12: return 0.3731763325901154f * z * (5.f * (z * z) - 3.f);
    case 13: return 0.45704579946446572f * x * (1.f - 5.f * (z * z));
    case 14: return 1.4453057213202769f * z * (x * x - y * y);
    default: return 0.59004358992664352f * x * (3.f * (y * y) - x * x);
    }
}

// One grid level as the lanes that encode it hold it. Both layouts keep a grid row along x in
// consecutive entries: dense levels are x-major, and a hashed level places row (y, z) at an offset
// in [0, table - side] drawn from a hash of (y, z) (multiply-high range reduction), so one 16-byte
// load fetches the two entries of an x-edge of a cell.
struct GridLevel {
    const uint2* table;
    float res;
    int last;             // the last cell along an axis
    uint32_t side, span;  // entries along an axis; row offsets (side <= table is checked at create)
    bool dense;
};

__device__ __forceinline__ GridLevel grid_level(const GuideNet& net, int l) {
    const uint32_t res = net.res[l];
    const uint64_t side = uint64_t(res) + 1;
    return GridLevel{reinterpret_cast<const uint2*>(net.grid) + size_t(l) * net.table, float(res), int(res) - 1,
                     uint32_t(side), net.table - uint32_t(side) + 1u, side * side * side <= uint64_t(net.table)};
}

// One of those corners: its table index and weight.
__device__ __forceinline__ void grid_corner(uint32_t table, uint32_t res, const float pn[3], int cx, int cy, int cz,
                                            uint32_t& idx, float& w) {
    int ci[3];
    float fr[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float x = pn[a] * float(res);
        int c = int(floorf(x));
        c = c >= int(res) ? int(res) - 1 : (c < 0 ? 0 : c);
        ci[a] = c;
        fr[a] = x - float(c);
    }
    const uint32_t ix = uint32_t(ci[0] + cx), iy = uint32_t(ci[1] + cy), iz = uint32_t(ci[2] + cz);
    const uint64_t side = uint64_t(res) + 1;
    const bool dense = side * side * side <= uint64_t(table);
    const uint32_t span = table - uint32_t(side) + 1u;
    idx = dense ? ix + uint32_t(side) * (iy + uint32_t(side) * iz)
                : uint32_t((uint64_t((iy * 2654435761u) ^ (iz * 805459861u)) * span) >> 32) + ix;
    const float wx = cx ? fr[0] : 1.f - fr[0];
    const float wy = cy ? fr[1] : 1.f - fr[1];
    const float wz = cz ? fr[2] : 1.f - fr[2];
    w = (wx * wy) * wz;
}

__device__ __forceinline__ void normalise(const GuideNet& net, f3 p, float pn[3]) {
    pn[0] = fminf(1.f, fmaxf(0.f, (p.x - net.offset[0]) * net.scale[0]));
    pn[1] = fminf(1.f, fmaxf(0.f, (p.y - net.offset[1]) * net.scale[1]));
    pn[2] = fminf(1.f, fmaxf(0.f, (p.z - net.offset[2]) * net.scale[2]));
}

// Entries i and i + 1 of one level's table (the two x-corners of a cell edge, G_FEATS fp16
// features each) in one 16-byte load (8-byte aligned).
struct __attribute__((packed, aligned(8))) EntryPair {
    uint32_t a0, a1, b0, b1;
};
static_assert(G_FEATS == 4, "one entry = two 32-bit words");

// Grid levels of lane group g: chunk-0 slots s < 4 hold features 4g + s (level g), slots s >= 4
// hold features 16 + 4g + s - 4 (level 4 + g), as feat_of(0, g, s) = G_FEATS * level + feature.
__device__ __forceinline__ int slot_level(int g, int h) { return 4 * h + g; }

__device__ __forceinline__ void add_entry(float f[4], float w, uint32_t lo, uint32_t hi) {
    f[0] += w * half_to_float(uint16_t(lo & 0xFFFFu));
    f[1] += w * half_to_float(uint16_t(lo >> 16));
    f[2] += w * half_to_float(uint16_t(hi & 0xFFFFu));
    f[3] += w * half_to_float(uint16_t(hi >> 16));
}

// The four features of one grid level at normalised position pn: trilinear over the cell's corners.
// The rows of the four x-edges are computed once for both of their corners, in 32 bits (a dense
// level's indices are below the table's size).
__device__ __forceinline__ void encode_level(const GridLevel& L, const float pn[3], _Float16 out[G_FEATS]) {
    uint32_t ci[3];
    float fr[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float x = pn[a] * L.res;
        const int c = min(max(int(floorf(x)), 0), L.last);
        ci[a] = uint32_t(c);
        fr[a] = x - float(c);
    }
    const uint32_t hy = ci[1] * 2654435761u, hz = ci[2] * 805459861u;
    const uint32_t row = L.side * (ci[1] + L.side * ci[2]), up = L.side * L.side;
    const float wx[2] = {1.f - fr[0], fr[0]}, wy[2] = {1.f - fr[1], fr[1]}, wz[2] = {1.f - fr[2], fr[2]};
    float f[G_FEATS] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t y = e & 1, z = e >> 1;
        const uint32_t hashed = __umulhi((hy + y * 2654435761u) ^ (hz + z * 805459861u), L.span);
        const uint32_t dense = row + (y ? L.side : 0u) + (z ? up : 0u);
        const EntryPair v = *reinterpret_cast<const EntryPair*>(L.table + ((L.dense ? dense : hashed) + ci[0]));
        add_entry(f, (wx[0] * wy[y]) * wz[z], v.a0, v.a1);
        add_entry(f, (wx[1] * wy[y]) * wz[z], v.b0, v.b1);
    }
#pragma unroll
    for (int k = 0; k < G_FEATS; k++) out[k] = _Float16(f[k]);
}

// Encoding of one query by lane group g: chunk 0 = grid levels g and 4 + g (four features
// each), chunk 1 = SH coefficients 4g..4g+3, then zeros.
__device__ __forceinline__ void encode(const GuideNet& net, f3 p, f3 wo, int g, half8_t x[2]) {
    float pn[3];
    normalise(net, p, pn);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        _Float16 f[G_FEATS];
        encode_level(grid_level(net, slot_level(g, h)), pn, f);
#pragma unroll
        for (int k = 0; k < G_FEATS; k++) x[0][4 * h + k] = f[k];
    }
#pragma unroll
    for (int s = 0; s < 4; s++) x[1][s] = _Float16(sh_coef(4 * g + s, wo.x, wo.y, wo.z));
#pragma unroll
    for (int s = 4; s < 8; s++) x[1][s] = _Float16(0.f);
}

// acc[t][ot] = W_layer (rows 16 ot..) * x[t] for ot < OT and each of the T tiles.
template <int OT, int T = NT>
__device__ __forceinline__ void layer_mfma(const half8_t* frag, int layer, const half8_t (&x)[T][2],
                                           floatx4 (&acc)[T][4], int lane) {
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int ot = 0; ot < 4; ot++) acc[t][ot] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
        for (int ot = 0; ot < OT; ot++) {
            const half8_t a = frag[((layer * 4 + ot) * 2 + c) * 64 + lane];
#pragma unroll
            for (int t = 0; t < T; t++) acc[t][ot] = mfma(a, x[t][c], acc[t][ot]);
        }
    }
}

// D layout -> B operand of the next layer (fp16, ReLU). The maximum is taken of the converted pairs:
// the same values as before the conversion, in a quarter of the instructions.
template <int T = NT>
__device__ __forceinline__ void relu_to_operand(const floatx4 (&acc)[T][4], half8_t (&x)[T][2]) {
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int s = 0; s < 8; s++) x[t][c][s] = _Float16(acc[t][2 * c + (s >> 2)][s & 3]);
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int c = 0; c < 2; c++) x[t][c] = __builtin_elementwise_max(x[t][c], half8_t{});
}

// ---------------------------------------------------------------------------------------------
// inference

// Query sources: position and direction to the viewer of query i (false: no query).
struct QueueQueries {
    DeviceScene S;
    const float4 *qo, *qd, *hits;
    const uint32_t* count; // queue size on the device; null: n_fixed
    uint32_t n_fixed;
    __device__ __forceinline__ uint32_t n() const { return count ? *count : n_fixed; }
    __device__ __forceinline__ bool load(uint32_t i, f3& p, f3& wo) const {
        const float4 h = hits[i];
        const uint32_t gid = __float_as_uint(h.w);
        const float4 d = qd[i];
        wo = f3{-d.x, -d.y, -d.z};
        if (gid == 0xFFFFFFFFu) {
            p = f3{0.f, 0.f, 0.f};
            return false;
        }
        const float4* t = S.tri_shade + 4 * size_t(gid); // (p0, n0), (p1, n1), (p2, n2), ...
        const float4 a = t[0], b = t[1], c = t[2];
        const f3 p0{a.x, a.y, a.z};
        const f3 p1{b.x, b.y, b.z};
        const f3 p2{c.x, c.y, c.z};
        p = p0 + h.y * (p1 - p0) + h.z * (p2 - p0);
        return true;
    }
};
struct ArrayQueries {
    const float4 *pos, *wo;
    uint32_t count;
    __device__ __forceinline__ uint32_t n() const { return count; }
    __device__ __forceinline__ bool load(uint32_t i, f3& p, f3& w) const {
        const float4 a = pos[i], b = wo[i];
        p = f3{a.x, a.y, a.z};
        w = f3{b.x, b.y, b.z};
        return true;
    }
};

// Output rows of the inference kernels' last layer: lane group g (lanes 16g..16g+15) holds D rows
// 16 ot + 4 g + r (ot < 3, r < 4) of its query, so the last layer's rows are permuted when its
// weights are staged: slot k = 4 ot + r of group g computes output 10 g + k for k < 10 (lobes 2g
// and 2g+1, five outputs each), a zero row for k = 10, 11. Each lane then holds two whole
// lobes and no output has to move between lanes through LDS.
__device__ __forceinline__ int out_row_of(int row) {
    const int ot = row >> 4, g = (row & 15) >> 2, k = 4 * ot + (row & 3);
    return k < 10 ? 10 * g + k : -1;
}

// Sinks of one query's ten outputs held by lane group g: raw outputs or packed lobes. Every lane
// of the wave calls store (the lobe softmax reduces across the query's four lane groups).
struct RawSink {
    float* out;
    __device__ __forceinline__ void store(uint32_t i, bool valid, const float (&o)[10], int g) const {
        if (!valid) return;
#pragma unroll
        for (int k = 0; k < 10; k++) out[size_t(i) * G_OUT + 10 * g + k] = o[k];
    }
};
struct LobeSink {
    uint4* lobes;
    __device__ __forceinline__ void store(uint32_t i, bool valid, const float (&o)[10], int g) const {
        // softmax over the 8 lobe logits: two per lane, the other six in lanes +-16, +-32
        float zmax = fmaxf(o[0], o[5]);
        zmax = fmaxf(zmax, __shfl_xor(zmax, 16));
        zmax = fmaxf(zmax, __shfl_xor(zmax, 32));
        const float e0 = expf(o[0] - zmax), e1 = expf(o[5] - zmax);
        float sum = e0 + e1;
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (!valid) return;
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float pi = (h ? e1 : e0) / sum;
            const float kappa = expf(fminf(G_KAPPA_LOG_MAX, fmaxf(G_KAPPA_LOG_MIN, o[5 * h + 1])));
            f3 v{o[5 * h + 2], o[5 * h + 3], o[5 * h + 4]};
            const float len = sqrtf(dot(v, v));
            const f3 mu = len > 1e-6f ? v * (1.f / len) : f3{0.f, 0.f, 1.f};
            w[2 * h] = uint32_t(float_to_half(pi)) | (uint32_t(float_to_half(kappa)) << 16);
            w[2 * h + 1] = encode_normal(mu);
        }
        lobes[size_t(i) * 4 + g] = make_uint4(w[0], w[1], w[2], w[3]);
    }
};

// What the four lane groups need of a query, written by the one lane that read it.
struct __attribute__((aligned(16))) QueryRow {
    float pn[3]; // normalised position
    uint32_t valid;
    half8_t sh[2]; // 16 SH coefficients of the direction
};

// Inference: the forward weights in LDS (the last layer's rows permuted, out_row_of), 8 waves per
// block, one 16-query tile in registers at a time, and a query's outputs stay in the registers of the
// lanes that computed them. The grid is capped at the resident blocks (two per CU: 64 KB of LDS each),
// so the weights are staged once per block.
//
// Bound by the grid gathers' way through the L1 (the addresser is busy 4/5 of the time: eight 16-byte
// accesses per lane and tile) and, next, by the instructions issued; the matrix cores idle. What does
// not depend on the lane group is not repeated by it: a wave reads up to 64 queries at once, one per
// lane (position from the hit, normalisation, SH coefficients), and hands them to its tiles through LDS;
// the constants of a lane's two grid levels stay in registers. One bounce of a 960x540 16-spp frame
// takes 465 us, 525 with every lane group reading its queries and evaluating its own coefficients in a
// divergent switch. More waves per SIMD (five, six) and mixed-precision FMAs in place of the
// conversions of the gathered halves change nothing.
template <class Q, class Sink>
__global__ __launch_bounds__(IB) __attribute__((amdgpu_waves_per_eu(4))) void k_guide_infer(GuideNet net, Q q, Sink sink) {
    __shared__ half8_t frag[G_FRAGS * 64]; // 40 KB: forward fragments of all layers
    __shared__ QueryRow queries[IW][16 * I_TILES];
    for (int k = threadIdx.x; k < G_FRAGS * 64; k += IB) {
        const int layer = k / (8 * 64);
        if (layer < G_LAYERS - 1) {
            frag[k] = net.frag_fwd[k];
        } else {
            // [layer][ot][c][lane']: lane' = 16 kg + rr holds row 16 ot + rr of k-group kg
            const int ot = (k >> 7) & 3, c = (k >> 6) & 1, l = k & 63;
            const int o = out_row_of(16 * ot + (l & 15));
            frag[k] = o < 0 ? half8_t{} : net.frag_fwd[((layer * 4 + (o >> 4)) * 2 + c) * 64 + (l & ~15) + (o & 15)];
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const uint32_t n = q.n();
    // tiles per wave iteration: the fewest iterations of up to I_TILES, then spread evenly over them
    const uint32_t waves = gridDim.x * IW;
    const uint32_t rounds = (n / 16 + (n % 16 != 0) + waves - 1) / waves;
    const uint32_t iterations = max((rounds + I_TILES - 1) / I_TILES, 1u);
    const uint32_t tiles = max((rounds + iterations - 1) / iterations, 1u);
    const GridLevel levels[2] = {grid_level(net, slot_level(g, 0)), grid_level(net, slot_level(g, 1))};
    QueryRow* rows = queries[wave];
    const uint32_t stride = waves * 16 * tiles;
    for (uint32_t base = (blockIdx.x * IW + wave) * 16 * tiles; base < n; base += stride) { // wave-uniform
        {
            const uint32_t i = base + lane;
            f3 p{0.f, 0.f, 0.f}, wo{0.f, 0.f, 1.f};
            QueryRow r;
            r.valid = uint32_t(lane) < 16 * tiles && i < n && q.load(i, p, wo);
            normalise(net, p, r.pn);
#pragma unroll
            for (int k = 0; k < 16; k++) {
                float c = sh_coef(k, wo.x, wo.y, wo.z);
                asm("" : "+v"(c)); // rounded to 32 bits first, as everywhere: no fused product and conversion
                r.sh[k >> 3][k & 7] = _Float16(c);
            }
            rows[lane] = r;
        }
        wave_lds_fence();
#pragma unroll 1
        for (uint32_t t = 0; t < tiles && base + 16 * t < n; t++) {
            const QueryRow& r = rows[16 * t + (lane & 15)];
            const float pn[3] = {r.pn[0], r.pn[1], r.pn[2]};
            const bool valid = r.valid != 0;
            half8_t x[1][2];
            floatx4 acc[1][4];
            _Float16 f[2][G_FEATS];
            encode_level(levels[0], pn, f[0]);
            encode_level(levels[1], pn, f[1]);
#pragma unroll
            for (int k = 0; k < 8; k++) x[0][0][k] = f[k >> 2][k & 3];
            const half4_t sh = reinterpret_cast<const half4_t*>(r.sh)[g];
            x[0][1] = half8_t{sh[0], sh[1], sh[2], sh[3], 0, 0, 0, 0};
#pragma unroll
            for (int layer = 0; layer < 4; layer++) {
                layer_mfma<4, 1>(frag, layer, x, acc, lane);
                relu_to_operand<1>(acc, x);
            }
            layer_mfma<3, 1>(frag, 4, x, acc, lane);
            float o[10];
#pragma unroll
            for (int k = 0; k < 10; k++) o[k] = acc[0][k >> 2][k & 3];
            sink.store(base + 16 * t + (lane & 15), valid, o, g);
        }
        wave_lds_fence(); // the tiles have read their rows
    }
}

// ---------------------------------------------------------------------------------------------
// training

// Sums of the record weights by G_SUM_BLOCKS blocks, each in a fixed order; weight_sum adds them.
// One block alone took 24 us for 65,536 records (one wave in flight per SIMD of one CU).
__global__ __launch_bounds__(256) void k_guide_sum_weights(const float4* __restrict__ rec, uint32_t n,
                                                           float* __restrict__ scalars) {
    __shared__ float part[4];
    float s = 0.f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) s += rec[3 * size_t(i)].w;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        scalars[1 + blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
        if (blockIdx.x == 0) scalars[0] = 0.f;
    }
}
__device__ __forceinline__ float weight_sum(const float* __restrict__ scalars, int lane) {
    static_assert(G_SUM_BLOCKS == 64, "one partial sum per lane");
    float s = scalars[1 + lane];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    return s;
}

// Stores the 8 fp16 values of a B operand (features feat_of(c, g, s)) of record r.
__device__ __forceinline__ void store_operand(_Float16* base, uint32_t r, int g, const half8_t x[2]) {
    _Float16* row = base + size_t(r) * G_WIDTH;
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
            half4_t v{x[c][4 * h], x[c][4 * h + 1], x[c][4 * h + 2], x[c][4 * h + 3]};
            *reinterpret_cast<half4_t*>(row + 16 * (2 * c + h) + 4 * g) = v;
        }
}

// d(-log q)/d(outputs) of one record for lobes 4*half_ .. 4*half_+3 (their 20 outputs in o), scaled
// by s; returns -log q. The two lanes of a record, lane bit 0 = half_, both call this: the softmax
// and the mixture's density are reduced across the pair.
__device__ __forceinline__ float lobe_gradient(const float* o, f3 d, float s, float (&g)[20]) {
    constexpr int N = G_LOBES / 2;
    float zmax = fmaxf(fmaxf(o[0], o[5]), fmaxf(o[10], o[15]));
    zmax = fmaxf(zmax, __shfl_xor(zmax, 1));
    float e[N], esum = 0.f;
#pragma unroll
    for (int k = 0; k < N; k++) {
        e[k] = expf(o[5 * k] - zmax);
        esum += e[k];
    }
    esum += __shfl_xor(esum, 1);
    float pi[N], kap[N], f[N], cm[N], len[N], q = 0.f;
    f3 mu[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        pi[k] = e[k] / esum;
        kap[k] = expf(fminf(G_KAPPA_LOG_MAX, fmaxf(G_KAPPA_LOG_MIN, o[5 * k + 1])));
        const f3 v{o[5 * k + 2], o[5 * k + 3], o[5 * k + 4]};
        len[k] = sqrtf(dot(v, v));
        mu[k] = len[k] > 1e-6f ? v * (1.f / len[k]) : f3{0.f, 0.f, 0.f};
        cm[k] = dot(mu[k], d);
        f[k] = kap[k] / (6.2831853071795864f * -expm1f(-2.f * kap[k])) * expf(kap[k] * (cm[k] - 1.f));
        q += pi[k] * f[k];
    }
    q += __shfl_xor(q, 1);
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float r = pi[k] * f[k] / q;
        const float kk = kap[k], z = o[5 * k + 1];
        const bool clamped = z < G_KAPPA_LOG_MIN || z > G_KAPPA_LOG_MAX;
        const float dlogf = 1.f / kk - 2.f / expm1f(2.f * kk) + (cm[k] - 1.f);
        const bool dir = len[k] > 1e-6f;
        g[5 * k] = s * (pi[k] - r);
        g[5 * k + 1] = clamped ? 0.f : s * (-r * dlogf * kk);
        g[5 * k + 2] = dir ? s * (-r * kk * (d.x - cm[k] * mu[k].x) / len[k]) : 0.f;
        g[5 * k + 3] = dir ? s * (-r * kk * (d.y - cm[k] * mu[k].y) / len[k]) : 0.f;
        g[5 * k + 4] = dir ? s * (-r * kk * (d.z - cm[k] * mu[k].z) / len[k]) : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 20; k++) g[k] = q > 0.f ? fminf(G_DOUT_CLAMP, fmaxf(-G_DOUT_CLAMP, g[k])) : 0.f;
    return q > 0.f ? -logf(q) : 0.f;
}

// Adds the grid gradient of up to WQ records (rows of `enc`: 32 gradients at the encoding as
// [level][feature], then the normalised position) to grid_grad.
//
// Eight lanes cover one cell edge along x, whose two entries are adjacent in the table: 2 x 4
// 64-bit counters, 64 consecutive bytes. A wave's atomic instruction so touches 8 edges (four
// edges of a cell, two levels) in 8 line segments. With one lane per (record, level) and its 32
// counters added one instruction after the other every lane hit a line of its own, and the L2's
// atomic request rate bound the kernel: 671 us for 65,536 records.
__device__ __forceinline__ void scatter_grid_gradient(const GuideNet& net, const float (*enc)[48], uint32_t first,
                                                      uint32_t n, int lane, unsigned long long* __restrict__ grid_grad) {
    const int k = lane & 3, cx = (lane >> 2) & 1, cy = (lane >> 3) & 1, cz = (lane >> 4) & 1, lh = lane >> 5;
    const uint32_t rows = first < n ? min(uint32_t(WQ), n - first) : 0u;
#pragma unroll
    for (int lp = 0; lp < G_LEVELS / 2; lp++) {
        const int l = 2 * lp + lh;
        const uint32_t res = lh ? net.res[2 * lp + 1] : net.res[2 * lp];
        unsigned long long* table = grid_grad + size_t(l) * net.table * G_FEATS + k;
#pragma unroll 2
        for (uint32_t q = 0; q < rows; q++) {
            const float* e = enc[q];
            uint32_t idx;
            float w;
            grid_corner(net.table, res, e + G_FEATS * G_LEVELS, cx, cy, cz, idx, w);
            const float v = w * e[G_FEATS * l + k];
            // non-finite contributions are dropped (they would poison Adam's moments)
            if (v != 0.f && fabsf(v) < __builtin_inff()) {
                const float cv = fminf(fmaxf(v, -G_GRID_FX_CLAMP), G_GRID_FX_CLAMP);
                atomicAdd(table + size_t(idx) * G_FEATS, (unsigned long long)__float2ll_rn(cv * G_GRID_FX));
            }
        }
    }
}

// Forward and backward of BQ records per block iteration: stores every layer's input (H) and
// output gradient (D) for the weight-gradient GEMM and adds the grid gradient. The backward pass
// needs of a layer's input only which activations were positive: one bit each, instead of the
// inputs of all layers in registers (444 registers and scratch, one wave per SIMD).
__global__ __launch_bounds__(GB) __attribute__((amdgpu_waves_per_eu(2))) void k_guide_fwd_bwd(
    GuideNet net, const float4* __restrict__ rec, uint32_t n, GuideTrainBuffers B) {
    // rows of a record: the outputs, then their gradients, then the gradient at the encoding
    __shared__ float outs[4][WQ][48];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const float mean_w = weight_sum(B.scalars, lane) / float(n > 0 ? n : 1);
    for (uint32_t base = blockIdx.x * BQ; base < n; base += gridDim.x * BQ) {
        half8_t x[NT][2];
        floatx4 acc[NT][4];
        uint32_t rid[NT];
        uint64_t active[NT] = {}; // bit 16 k + 8 c + s: input (c, s) of layer 1 + k is positive
#pragma unroll
        for (int t = 0; t < NT; t++) {
            rid[t] = base + wave * WQ + t * 16 + (lane & 15);
            f3 p{0.f, 0.f, 0.f}, wo{0.f, 0.f, 1.f};
            if (rid[t] < n) {
                const float4 a = rec[3 * size_t(rid[t])], b = rec[3 * size_t(rid[t]) + 1];
                p = f3{a.x, a.y, a.z};
                wo = f3{b.x, b.y, b.z};
            }
            encode(net, p, wo, g, x[t]);
            if (rid[t] < n) store_operand(B.H, rid[t], g, x[t]);
        }
#pragma unroll 1
        for (int layer = 0; layer < 4; layer++) {
            layer_mfma<4>(net.frag_fwd, layer, x, acc, lane);
            relu_to_operand(acc, x);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                uint32_t m = 0;
#pragma unroll
                for (int c = 0; c < 2; c++)
#pragma unroll
                    for (int s = 0; s < 8; s++) m |= float(x[t][c][s]) > 0.f ? 1u << (8 * c + s) : 0u;
                active[t] |= uint64_t(m) << (16 * layer);
                if (rid[t] < n) store_operand(B.H + size_t(layer + 1) * B.cap * G_WIDTH, rid[t], g, x[t]);
            }
        }
        layer_mfma<3>(net.frag_fwd, 4, x, acc, lane);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int ot = 0; ot < 3; ot++)
#pragma unroll
                for (int r = 0; r < 4; r++) outs[wave][t * 16 + (lane & 15)][16 * ot + 4 * g + r] = acc[t][ot][r];
        __syncthreads();
        {
            const int qi = lane >> 1, half_ = lane & 1;
            const uint32_t i = base + wave * WQ + qi;
            const bool valid = i < n;
            float o[20], gr[20];
#pragma unroll
            for (int k = 0; k < 20; k++) o[k] = outs[wave][qi][20 * half_ + k];
            f3 dir{0.f, 0.f, 1.f};
            float s = 0.f;
            if (valid) {
                const float4 a = rec[3 * size_t(i)], c = rec[3 * size_t(i) + 2];
                s = mean_w > 0.f ? fminf(G_WEIGHT_SCALE_MAX, a.w / mean_w) : 0.f;
                dir = f3{c.x, c.y, c.z};
            }
            const float nlq = lobe_gradient(o, dir, s, gr);
            __syncthreads(); // every output is in registers: the rows now take the gradients
#pragma unroll
            for (int k = 0; k < 20; k++) outs[wave][qi][20 * half_ + k] = valid ? gr[k] : 0.f;
            if (half_ == 1)
#pragma unroll
                for (int k = 40; k < 48; k++) outs[wave][qi][k] = 0.f;
            // loss: one lane per record, one atomic per wave
            float l = (half_ == 0 && valid) ? s * nlq : 0.f;
            for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
            if (lane == 0) atomicAdd(B.scalars, l);
        }
        __syncthreads();
        // gradient at the outputs as B operand (features >= 48 are zero)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const int fo = feat_of(c, g, s);
                    x[t][c][s] = _Float16(fo < 48 ? outs[wave][t * 16 + (lane & 15)][fo] : 0.f);
                }
#pragma unroll 1
        for (int layer = 4; layer >= 0; layer--) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (rid[t] < n) store_operand(B.D + size_t(layer) * B.cap * G_WIDTH, rid[t], g, x[t]);
            layer_mfma<4>(net.frag_bwd, layer, x, acc, lane); // acc = W^T d: gradient at the layer's input
            if (layer > 0) {
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const uint32_t m = uint32_t(active[t] >> (16 * (layer - 1)));
#pragma unroll
                    for (int c = 0; c < 2; c++)
#pragma unroll
                        for (int s = 0; s < 8; s++)
                            x[t][c][s] = _Float16((m >> (8 * c + s)) & 1u ? acc[t][2 * c + (s >> 2)][s & 3] : 0.f);
                }
            }
        }
        // acc = gradient at the encoding: in-tile 0 holds features 4g+r (level g), in-tile 1
        // holds 16+4g+r (level 4+g). It goes through LDS (the output rows, read for the last time
        // above) so that the lanes of one atomic instruction cover whole cell edges.
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float* o = outs[wave][t * 16 + (lane & 15)];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int k = 0; k < G_FEATS; k++) o[G_FEATS * slot_level(g, h) + k] = acc[t][h][k];
            if (g == 0 && rid[t] < n) {
                const float4 a = rec[3 * size_t(rid[t])];
                normalise(net, f3{a.x, a.y, a.z}, o + G_FEATS * G_LEVELS);
            }
        }
        __syncthreads();
        scatter_grid_gradient(net, outs[wave], base + wave * WQ, n, lane, B.grid_grad);
    }
}

// dW_layer = sum over records of D_layer (outputs) x H_layer (inputs): per block a range of
// G_WGRAD_RECORDS records, staged 32 at a time through LDS as [feature][record]; wave w
// computes output rows 16w..16w+15 for all 64 inputs.
__global__ __launch_bounds__(GB) void k_guide_wgrad(GuideTrainBuffers B, uint32_t n) {
    __shared__ __attribute__((aligned(16))) _Float16 Dt[64][40]; // rows of 80 bytes: 16-byte aligned reads
    __shared__ __attribute__((aligned(16))) _Float16 Ht[64][40];
    const int layer = blockIdx.y, kb = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const _Float16* D = B.D + size_t(layer) * B.cap * G_WIDTH;
    const _Float16* H = B.H + size_t(layer) * B.cap * G_WIDTH;
    const uint32_t r0 = kb * G_WGRAD_RECORDS;
    const uint32_t r1 = min(n, r0 + G_WGRAD_RECORDS);
    floatx4 acc[4];
    for (int it = 0; it < 4; it++) acc[it] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (uint32_t rb = r0; rb < r1; rb += 32) {
        {
            const int r = threadIdx.x >> 3, f0 = (threadIdx.x & 7) * 8;
            const uint32_t rr = rb + r;
            half8_t dv = {}, hv = {};
            if (rr < r1) {
                dv = *reinterpret_cast<const half8_t*>(D + size_t(rr) * G_WIDTH + f0);
                hv = *reinterpret_cast<const half8_t*>(H + size_t(rr) * G_WIDTH + f0);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                Dt[f0 + j][r] = dv[j];
                Ht[f0 + j][r] = hv[j];
            }
        }
        __syncthreads();
        const half8_t a = *reinterpret_cast<const half8_t*>(&Dt[16 * wave + (lane & 15)][8 * g]);
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const half8_t b = *reinterpret_cast<const half8_t*>(&Ht[16 * it + (lane & 15)][8 * g]);
            acc[it] = mfma(a, b, acc[it]);
        }
        __syncthreads();
    }
    float* P = B.partials + (size_t(layer) * B.kblocks + kb) * G_WIDTH * G_WIDTH;
#pragma unroll
    for (int it = 0; it < 4; it++)
#pragma unroll
        for (int r = 0; r < 4; r++) P[(16 * wave + 4 * g + r) * G_WIDTH + 16 * it + (lane & 15)] = acc[it][r];
}

// Sum over the blocks' partials of weight element e, by the four waves of a block of GB threads
// (64 elements per block; wave w takes every fourth partial from w on); valid in wave 0. Every
// thread of the block calls this.
constexpr int WSUM_ELEMS = 64;
__device__ __forceinline__ float wgrad_sum(const GuideTrainBuffers& B, uint32_t e) {
    __shared__ float part[4][WSUM_ELEMS];
    const uint32_t layer = e / (G_WIDTH * G_WIDTH), k = e % (G_WIDTH * G_WIDTH), wave = threadIdx.x >> 6;
    const float* p = B.partials + size_t(layer) * B.kblocks * G_WIDTH * G_WIDTH + k;
    float s = 0.f;
    for (uint32_t kb = wave; kb < B.kblocks; kb += 4) s += p[size_t(kb) * G_WIDTH * G_WIDTH];
    part[wave][threadIdx.x & 63] = s;
    __syncthreads();
    const uint32_t c = threadIdx.x & 63;
    return (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

__global__ __launch_bounds__(GB) void k_guide_reduce_wgrad(GuideTrainBuffers B, float* __restrict__ dW) {
    const uint32_t e = blockIdx.x * WSUM_ELEMS + (threadIdx.x & 63);
    const float s = wgrad_sum(B, e);
    if (threadIdx.x < WSUM_ELEMS) dW[e] = s;
}

// Fragment positions of weight W_layer[o][i]: forward (A = W) and backward (A = W^T).
__device__ __forceinline__ void frag_positions(int layer, int o, int i, uint32_t& fwd, int& fs, uint32_t& bwd, int& bs) {
    {
        const int ti = i >> 4, c = ti >> 1, g = (i & 15) >> 2;
        fs = 4 * (ti & 1) + (i & 3);
        fwd = uint32_t(((layer * 4 + (o >> 4)) * 2 + c) * 64 + 16 * g + (o & 15));
    }
    {
        const int to = o >> 4, c = to >> 1, g = (o & 15) >> 2;
        bs = 4 * (to & 1) + (o & 3);
        bwd = uint32_t(((layer * 4 + (i >> 4)) * 2 + c) * 64 + 16 * g + (i & 15));
    }
}

__global__ __launch_bounds__(GB) void k_guide_adam_w(GuideParams p, GuideTrainBuffers B, float lr, float scale,
                                                     float bc1, float bc2, int update) {
    const uint32_t e = blockIdx.x * WSUM_ELEMS + (threadIdx.x & 63);
    const float gsum = update ? wgrad_sum(B, e) : 0.f;
    if (threadIdx.x >= WSUM_ELEMS) return;
    const int layer = int(e / (G_WIDTH * G_WIDTH)), o = int((e / G_WIDTH) % G_WIDTH), i = int(e % G_WIDTH);
    float w = p.w[e];
    if (update && !(layer == G_LAYERS - 1 && o >= G_OUT)) {
        const float gr = gsum * scale;
        const float m = 0.9f * p.w_m[e] + 0.1f * gr;
        const float v = 0.99f * p.w_v[e] + 0.01f * gr * gr;
        p.w_m[e] = m;
        p.w_v[e] = v;
        w -= lr * (m / bc1) / (sqrtf(v / bc2) + 1e-10f);
        p.w[e] = w;
    }
    uint32_t fwd, bwd;
    int fs, bs;
    frag_positions(layer, o, i, fwd, fs, bwd, bs);
    reinterpret_cast<_Float16*>(p.frag_fwd + fwd)[fs] = _Float16(w);
    reinterpret_cast<_Float16*>(p.frag_bwd + bwd)[bs] = _Float16(w);
}

__global__ void k_guide_adam_grid(GuideParams p, unsigned long long* __restrict__ grad, float lr, float scale,
                                  float bc1, float bc2, int update) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < p.grid_count; e += stride) {
        float w = p.g[e];
        if (update) {
            const float gr = float((long long)grad[e]) * (1.f / G_GRID_FX) * scale;
            grad[e] = 0ull;
            float m = p.g_m[e], v = p.g_v[e];
            if (gr != 0.f || m != 0.f) {
                m = 0.9f * m + 0.1f * gr;
                v = 0.99f * v + 0.01f * gr * gr;
                p.g_m[e] = m;
                p.g_v[e] = v;
                w -= lr * (m / bc1) / (sqrtf(v / bc2) + 1e-10f);
                p.g[e] = w;
            }
        }
        p.grid[e] = _Float16(w);
    }
}

// Sort keys (the third float4's w of each record) and their record indices.
__global__ void k_guide_record_keys(const float4* __restrict__ in, uint32_t n, uint32_t* __restrict__ keys,
                                    uint32_t* __restrict__ vals) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += stride) {
        keys[r] = __float_as_uint(in[3 * size_t(r) + 2].w);
        vals[r] = r;
    }
}

// Record k of the sorted order -> slot (k * 2654435761) mod n (2654435761 is prime and n < 2^32,
// so the map is a permutation); the key is cleared.
__global__ void k_guide_record_place(const float4* __restrict__ in, const uint32_t* __restrict__ order, uint32_t n,
                                     float4* __restrict__ out) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
        const float4* a = in + 3 * size_t(order[k]);
        float4* b = out + 3 * ((uint64_t(k) * 2654435761ull) % n);
        const float4 c = a[2];
        b[0] = a[0];
        b[1] = a[1];
        b[2] = make_float4(c.x, c.y, c.z, 0.f);
    }
}

int blocks_for(uint64_t n, int per_block, int cap) {
    const uint64_t b = (n + per_block - 1) / per_block;
    return int(b < uint64_t(cap) ? (b > 0 ? b : 1) : cap);
}

} // namespace

hipError_t launch_guide_infer_queue(const GuideNet& net, const DeviceScene& s, const float4* qo, const float4* qd,
                                    const float4* hits, const uint32_t* count, uint32_t n_max, uint4* lobes,
                                    hipStream_t st) {
    if (n_max == 0) return hipSuccess;
    const QueueQueries q{s, qo, qd, hits, count, n_max};
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_guide_infer<QueueQueries, LobeSink>), dim3(blocks_for(n_max, 16 * IW, 512)),
                       dim3(IB), 0, st, net, q, LobeSink{lobes});
    return hipGetLastError();
}

hipError_t launch_guide_forward(const GuideNet& net, const float4* pos, const float4* wo, uint32_t n, float* out,
                                hipStream_t st) {
    if (n == 0) return hipSuccess;
    const ArrayQueries q{pos, wo, n};
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_guide_infer<ArrayQueries, RawSink>), dim3(blocks_for(n, 16 * IW, 512)), dim3(IB),
                       0, st, net, q, RawSink{out});
    return hipGetLastError();
}

hipError_t launch_guide_gradient(const GuideNet& net, const float4* records, uint32_t n, GuideTrainBuffers& b,
                                 hipStream_t st) {
    if (n > b.cap) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_guide_sum_weights, dim3(G_SUM_BLOCKS), dim3(256), 0, st, records, n, b.scalars);
    if (n == 0) return hipGetLastError();
    hipLaunchKernelGGL(k_guide_fwd_bwd, dim3(blocks_for(n, BQ, 1024)), dim3(GB), 0, st, net, records, n, b);
    const uint32_t kb = (n + G_WGRAD_RECORDS - 1) / G_WGRAD_RECORDS;
    if (kb > b.kblocks) return hipErrorInvalidValue;
    // the partials are laid out for exactly kb blocks; the reductions read the same layout
    b.kblocks = kb;
    hipLaunchKernelGGL(k_guide_wgrad, dim3(kb, G_LAYERS), dim3(GB), 0, st, b, n);
    return hipGetLastError();
}

hipError_t launch_guide_reduce_wgrad(const GuideTrainBuffers& b, float* dW, hipStream_t st) {
    hipLaunchKernelGGL(k_guide_reduce_wgrad, dim3(G_LAYERS * G_WIDTH * G_WIDTH / WSUM_ELEMS), dim3(GB), 0, st, b, dW);
    return hipGetLastError();
}

hipError_t launch_guide_adam(const GuideParams& p, const GuideTrainBuffers& b, float lr, float scale, float bc1,
                             float bc2, hipStream_t st) {
    hipLaunchKernelGGL(k_guide_adam_w, dim3(G_LAYERS * G_WIDTH * G_WIDTH / WSUM_ELEMS), dim3(GB), 0, st, p, b, lr,
                       scale, bc1, bc2, 1);
    hipLaunchKernelGGL(k_guide_adam_grid, dim3(blocks_for(p.grid_count, 256, 8192)), dim3(256), 0, st, p, b.grid_grad,
                       lr, scale, bc1, bc2, 1);
    return hipGetLastError();
}

hipError_t launch_guide_pack(const GuideParams& p, hipStream_t st) {
    GuideTrainBuffers none{};
    hipLaunchKernelGGL(k_guide_adam_w, dim3(G_LAYERS * G_WIDTH * G_WIDTH / WSUM_ELEMS), dim3(GB), 0, st, p, none,
                       0.f, 0.f, 1.f, 1.f, 0);
    hipLaunchKernelGGL(k_guide_adam_grid, dim3(blocks_for(p.grid_count, 256, 8192)), dim3(256), 0, st, p, nullptr,
                       0.f, 0.f, 1.f, 1.f, 0);
    return hipGetLastError();
}

size_t launch_guide_order_temp_bytes(uint32_t cap) {
    size_t bytes = 0;
    if (rocprim::radix_sort_pairs(nullptr, bytes, static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                  static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), cap, 0u, 32u) !=
        hipSuccess)
        return 0;
    return bytes;
}

hipError_t launch_guide_order_records(const float4* in, uint32_t n, uint32_t* keys, uint32_t* vals, void* temp,
                                      size_t temp_bytes, float4* out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const int g = blocks_for(n, 256, 4096);
    hipLaunchKernelGGL(k_guide_record_keys, dim3(g), dim3(256), 0, st, in, n, keys, vals);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t bytes = temp_bytes;
    e = rocprim::radix_sort_pairs(temp, bytes, keys, keys + n, vals, vals + n, n, 0u, 32u, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_guide_record_place, dim3(g), dim3(256), 0, st, in, vals + n, n, out);
    return hipGetLastError();
}

} // namespace mrt

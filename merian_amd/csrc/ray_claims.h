// How the waves of a persistent trace launch divide a caller's rays among work cursors.
//
// One cursor takes 75 to 120 M claims a second whichever waves make them, and a launch of cheap rays
// ends with thousands of claims of 64; eight cursors in cache lines of their own take 270 to 460 M.
// The rays go round the cursors in rows of CLAIM_ROW, so that the cursors' shares cost alike and no
// wave need look at another's: a wave belongs to one cursor, owns a part of its share and claims the
// rest (mrt_trace.h). Positions in a share are mapped to rays by claim_ray.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define MRT_CLAIMS_FN __host__ __device__ inline
#else
#define MRT_CLAIMS_FN inline
#endif

namespace mrt {

constexpr uint32_t CURSOR_BITS = 3;    // 2^CURSOR_BITS cursors
constexpr uint32_t CURSOR_STRIDE = 32; // words from one to the next: a 128-byte line each
constexpr uint32_t CURSOR_WORDS = CURSOR_STRIDE << CURSOR_BITS;
// 6 M camera rays in a million triangles: 4.31 ms with rows of 256, 4.41 with 1024, 4.35 with 4096; other
// arrays alike.
constexpr uint32_t CLAIM_ROW = 256;

struct RayClaims {
    uint32_t n;          // rays of the share
    uint32_t wave, waves; // this wave's number among the waves of its cursor
    uint32_t bits, home; // 2^bits cursors; the wave's own
};

// All n rays to one cursor.
MRT_CLAIMS_FN RayClaims one_cursor(uint32_t n, uint32_t wave, uint32_t waves) { return RayClaims{n, wave, waves, 0u, 0u}; }

// Shares of 2^CURSOR_BITS cursors for wave `w` of block `block` of `blocks`, `per_block` waves each.
// Consecutive blocks go to different XCDs, which differ in speed by a few percent: groups of
// 2^CURSOR_BITS consecutive blocks take one cursor, so that every cursor has blocks on every XCD (by
// XCD, 6 M incoherent rays in 200,000 triangles take 3.94 ms instead of 3.85). Launches of too few
// blocks for that have one cursor.
MRT_CLAIMS_FN RayClaims many_cursors(uint32_t n, uint32_t block, uint32_t blocks, uint32_t w, uint32_t per_block) {
    constexpr uint32_t B = CURSOR_BITS, C = 1u << B;
    if ((blocks >> (2u * B)) == 0u) return one_cursor(n, block * per_block + w, blocks * per_block);
    const uint32_t home = (block >> B) & (C - 1u);
    const uint32_t rows = n / CLAIM_ROW, last = rows & (C - 1u); // the cursor that has the row after the whole ones
    const uint32_t mine = ((rows >> B) + (home < last ? 1u : 0u)) * CLAIM_ROW + (home == last ? n % CLAIM_ROW : 0u);
    const uint32_t rest = blocks & (C * C - 1u); // blocks after the whole rounds of all cursors
    const uint32_t extra = rest > home * C ? (rest - home * C < C ? rest - home * C : C) : 0u;
    return RayClaims{mine, (((block >> (2u * B)) << B) + (block & (C - 1u))) * per_block + w,
                     (((blocks >> (2u * B)) << B) + extra) * per_block, B, home};
}

// Ray at position q of a share.
MRT_CLAIMS_FN uint32_t claim_ray(const RayClaims& c, uint32_t q) {
    return (((q / CLAIM_ROW) << c.bits) + c.home) * CLAIM_ROW + q % CLAIM_ROW;
}

} // namespace mrt

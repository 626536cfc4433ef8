// CPU check of merian_amd/csrc/ray_claims.h: over all waves of a launch, the parts of the shares that
// the waves own and the rest that they claim are every ray exactly once, whatever the ray count and
// the grid (rows that do not fill, blocks that do not make a whole round of the cursors).
#include "../../merian_amd/csrc/ray_claims.h"

#include <cstdio>
#include <map>
#include <vector>

using namespace mrt;

int main() {
    int failures = 0;
    const uint32_t counts[] = {1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 8193, 16383, 131071, 1000003};
    for (uint32_t n : counts)
        for (uint32_t blocks : {1u, 2u, 7u, 63u, 64u, 65u, 71u, 72u, 73u, 100u, 128u, 129u, 1000u})
            for (uint32_t per_block : {1u, 2u}) {
                std::vector<uint8_t> seen(n);
                std::map<uint32_t, std::vector<uint8_t>> ranks; // per cursor: waves by number
                std::map<uint32_t, RayClaims> share;
                bool bad = false;
                auto mark = [&](const RayClaims& c, uint32_t q) {
                    const uint32_t i = claim_ray(c, q);
                    if (i >= n || seen[i]++) bad = true;
                };
                for (uint32_t b = 0; b < blocks; b++)
                    for (uint32_t w = 0; w < per_block; w++) {
                        const RayClaims c = many_cursors(n, b, blocks, w, per_block);
                        std::vector<uint8_t>& r = ranks[c.home];
                        r.resize(c.waves);
                        if (c.wave >= c.waves || r[c.wave]++) bad = true;
                        if (share.count(c.home) && (share[c.home].n != c.n || share[c.home].waves != c.waves)) bad = true;
                        share[c.home] = c;
                        if (c.home >= (1u << c.bits) || c.home * CURSOR_STRIDE >= CURSOR_WORDS) bad = true;
                        const uint32_t own = (c.n / (2 * c.waves)) & ~63u;
                        for (uint32_t k = 0; k < own; k++) mark(c, c.wave * own + k);
                    }
                for (auto& h : share) {
                    const RayClaims& c = h.second;
                    for (uint8_t one : ranks[h.first]) bad |= one != 1;
                    for (uint32_t q = ((c.n / (2 * c.waves)) & ~63u) * c.waves; q < c.n; q++) mark(c, q);
                }
                if (share.size() != (share.begin()->second.bits ? 1u << CURSOR_BITS : 1u)) bad = true;
                for (uint8_t s : seen) bad |= s != 1;
                if (bad && failures++ < 10) std::printf("FAILED n %u blocks %u waves per block %u\n", n, blocks, per_block);
            }
    return failures ? 1 : 0;
}

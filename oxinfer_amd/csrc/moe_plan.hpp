// How a launch of the bf16 grouped expert matmuls (moe_bf16.hip) is cut into workgroups: arithmetic on sizes, no device code.
#pragma once
#include <cstddef>
#include <cstdint>

#include "formats.hpp"

namespace oxhip {

constexpr uint32_t MOE_PHASE = 16;  // steps x token tiles that a workgroup stages at a time

struct MoePlan {
    uint32_t rt;    // row tiles per wave
    uint32_t kw;    // waves that share the K steps of a group of row tiles
    uint32_t nrep;  // runs of 8 rt row tiles that a workgroup takes one after the other with one staging
    uint32_t nx;    // workgroups per chunk
};
// Chunks of up to 32 rows to be expected of a pass: an expert has a last one, half full on average, and its rows past 16 in 32s before it.
inline uint32_t moe_expected_chunks(size_t pairs, size_t n_exp) {
    return (uint32_t)((pairs < n_exp ? pairs : n_exp) + (pairs / n_exp > 16 ? (pairs - 16 * n_exp) / 32 : 0));
}
// The most that there can be.
inline size_t moe_most_chunks(size_t pairs, size_t n_exp) { return (pairs < n_exp ? pairs : n_exp) + pairs / 32 + 1; }
// `inter`: rows of the activation that the launch applies to its products (the gate / up launch), or 0; `chunks`: as many as are to be expected
// of the max_chunks there may be.
inline MoePlan moe_plan(int fmt, uint32_t n_out, uint32_t n_in, uint32_t inter, uint32_t max_chunks, uint32_t chunks) {
    const uint32_t nsteps = n_in / 128, tiles = inter ? inter / 16 : (n_out + 15) / 16;
    auto nx_of = [&](uint32_t r, uint32_t k) {
        const uint32_t per = (8 / k) * r / (inter ? 2 : 1);
        return (tiles + per - 1) / per;
    };
    // K over two or four waves where one wave per row would leave fewer workgroups than places. (The order of a sum's terms follows kw, and kw
    // the pass's size: the last bits of a token's result can differ with the number of tokens that share its pass.)
    uint32_t rt = 2, kw = 1;
    while (kw < 4 && nsteps / (2 * kw) >= 4 && (uint64_t)nx_of(rt, kw) * max_chunks < 512) kw *= 2;
    // Row tiles per wave, and runs of them that a workgroup takes one after the other with one staging (the down projection's rows fit a
    // phase): what takes fewer rounds of workgroups over the 512 places, a round as long as its waves' row tiles x steps and six more for its staging
    // and its end. At 256 tokens, MLX 4-bit: gate / up launch, two tiles and three, 128 experts of 2048 / 768 64.2 and 55.6 us (768 and 512
    // workgroups), 32 experts 38.9 and 48.5; down launch, one run of two tiles, of three, two, three and four of two, 128 experts 34.5, 36.3, 33.6, 38.0
    // and 34.4, 32 experts (two tiles, 320 workgroups) 23.4, 22.4, 24.9, 23.5 and 27.2. (Four row tiles spill in the form of two token tiles: 76.)
    // Over twelve shapes of 8 to 128 experts, 6 to 64 rows per expert and five formats (600 passes) the split so chosen costs a pass 2.0 % (gate / up)
    // and 0.7 % (down) over the best of all splits, 16 and 9 % at worst, where the rounds are just filled or just not.
    // The 16 items: `chunks` is high where experts have 17 to 24 rows, most of them in one chunk (136 for 128 at 18 rows), and would
    // otherwise count a round more than there is: 18 passes 3 to 26 % slower.
    uint32_t nrep = 1;
    if (kw == 1) {
        uint64_t least = ~0ull;
        for (uint32_t r = 2; r <= (fmt == FMT_Q8_0 ? 2u : 3u); r++)  // (Q8_0, a step being two records per row tile, keeps to two and one; three and several runs would spill)
            for (uint32_t n = 1; n <= (r == 2 && fmt != FMT_Q8_0 && !inter && 2 * nsteps <= MOE_PHASE ? 4u : 1u); n++) {
                const uint64_t items = (uint64_t)((nx_of(r, 1) + n - 1) / n) * chunks;
                const uint64_t cost = ((items > 16 ? items - 16 : 1) + 511) / 512 * (n * r * nsteps + 6);
                if (cost < least) {
                    least = cost;
                    rt = r;
                    nrep = n;
                }
            }
    }
    return {rt, kw, nrep, (nx_of(rt, kw) + nrep - 1) / nrep};
}

}  // namespace oxhip

// How the bf16 GEMMs (gemm.hip, gemm_short.hip) cut a product into workgroups and K slices: arithmetic on sizes, no device code.
#pragma once
#include <cstddef>
#include <cstdint>
#include <initializer_list>

#include "formats.hpp"

namespace oxhip {

constexpr uint32_t GEMM_WG_NT = 8;  // gemm.hip's row tiles per workgroup (128 rows), or 7 where that fills more CUs

// gemm.hip's token tiles per wave and waves per workgroup: one tile and four waves when the launch has at most four tiles (64 tokens), one
// tile and eight waves up to eight tiles (128 tokens), else two tiles and eight waves.
inline int gemm_nv(size_t mtiles) { return mtiles <= 8 ? 1 : 2; }
inline int gemm_waves(size_t mtiles) { return mtiles <= 4 ? 4 : 8; }

// Row tiles per workgroup (8, or 7 with two token tiles per wave) and K slices of a launch: the pair that costs least, in units
// of one K-step of an eight-tile workgroup (0.9 us with one token tile per wave, 1.2 to 1.5 us with two):
//   rounds of workgroups over the 256 CUs x K-steps per slice. Two workgroups with one token tile per wave share a CU and
//     take 1.55 steps' time for a step of each; a workgroup with two tiles per wave, or with eight waves of an 8-bit format, has
//     its CU to itself. A slice of four steps costs 4.65 (the pipeline fills as often): 5120 -> 2816, MLX 4-bit, 100 tokens 20.2 us
//     in 8 slices, 21.2 in 10.
//   1 for every million partial sums written and read back, 1.9 for those past six million, and 2 for the launch that adds them
//     (14336 -> 4096, MLX 4-bit, 420 tokens, 4 slices -> 8: 6.9 million more, as many steps, 63.6 -> 69.7 us).
// Any number of slices counts, not only powers of two. With two tiles: 14336 -> 4096, MLX 4-bit, 1100 tokens (160 workgroups) 167.6 us
// whole, 153.0 in 3 slices, 190.8 in 2; FP8 7168 x 18432 at 1100 tokens 397 us whole, 331 in 3. Four steps per slice at least
// (7168 -> 1536, Q8_0, 200 tokens: 30.7 us at 14 steps, 24.4 at 7, 23.5 at 5).
// Seven row tiles: 14336 rows x 512 tokens are one round of 256 workgroups of 112 rows instead of 224 of 128, 63 -> 60 us: a step of
// theirs costs 0.94 of one of eight, not 7/8 (counted as 7/8, 8192 rows x 512 tokens of 4096 columns went from 256 workgroups in two
// slices to 148 of seven tiles whole, Q4_K 46.5 -> 53.2 us; 7895 x 5888 at 224 tokens 37.1 -> 39.6).
struct GemmPlan {
    uint32_t nt, slices;
    double cost;
};
inline GemmPlan gemm_plan(int fmt, uint32_t n_out, uint32_t n_in, size_t mtiles) {
    const bool one = gemm_nv(mtiles) == 1;
    const uint32_t per_wg = gemm_waves(mtiles) * gemm_nv(mtiles), cols = (uint32_t)((mtiles + per_wg - 1) / per_wg);
    const uint32_t steps = (n_in + 127) / 128, tiles = (n_out + 15) / 16;
    const bool alone = !one || (gemm_waves(mtiles) == 8 && (fmt == FMT_Q8_0 || fmt == FMT_Q8F));
    // (Eight waves of one token tile: eight slices at most, 14336 -> 4096, MLX 4-bit at 70 tokens 29.1 us in 8 and 30.2 in 16.)
    const uint32_t most = one && gemm_waves(mtiles) == 8 ? 8 : 16;
    const double millions = (double)mtiles * 16 * n_out * 1e-6;
    auto sums = [](double m) { return m < 6 ? m : 6 + 1.9 * (m - 6); };
    GemmPlan best{GEMM_WG_NT, 1, 0};
    for (uint32_t nt : {GEMM_WG_NT, 7u}) {
        if (one && nt == 7) break;
        const uint64_t wgs = (uint64_t)((tiles + nt - 1) / nt) * cols;
        for (uint32_t z = 1; z <= most; z++) {
            const uint32_t per = (steps + z - 1) / z;
            if (z > 1 && steps / z < 4) break;
            // every slice must own a step: the kernel gives slice i the steps from i * per (33 steps in 8 slices of 5 would
            // start the last one past the end)
            if ((z - 1) * per >= steps) continue;
            const uint64_t rounds = (wgs * z + 255) / 256;
            const double held = alone ? (double)rounds : (double)(rounds / 2) * 1.55 + (double)(rounds % 2);
            const double cost = held * (per < 5 && z > 1 ? per + 0.65 : per) * (nt == 7 ? 0.94 : 1.0) + (z > 1 ? sums(z * millions) + 2 : 0);
            if ((nt == GEMM_WG_NT && z == 1) || cost < best.cost) best = GemmPlan{nt, z, cost};
        }
    }
    return best;
}

// Up to 64 tokens: gemm_short.hip's row tiles per workgroup and K slices, or gemm.hip's kernel of four waves (rt 0, slices as gemm_plan
// has them): what is expected to take least time. In microseconds, with the weights in HBM:
//   5.9, and 0.15 for every MB of weights;
//   gemm_short.hip: rounds of workgroups over the 256 CUs (two rounds count as 1.8 where two workgroups share a CU) x [0.166 + 0.168 per
//     matrix tile, for its start and the sums' way through LDS, + each wave's steps x (`row` per row tile: the records' way to operands;
//     `token` per token tile: the fragments' requests; `both` per matrix tile)] + 0.017 per step. K slices: 1.84 for the launch that adds
//     them and 2.46 for every million partial sums; 16 steps each, so that every wave has two.
//   gemm.hip: 0.97 + gemm_plan's units x `unit` + 1.09 per token tile + 0.03 more per MB.
// Constants by 48 shapes of 1000 to 36000 rows and 1500 to 18432 columns in ten formats and seven of up to 250000 rows in eight, at 24, 43 and 64
// tokens (FP8 40 and 64), every row tile count and up to four slices, weights in HBM and (the 48) in the Infinity Cache: single times to
// 4 to 10 %, what is taken 2 % above the best. Weights in the Infinity Cache come sooner, which favours few_tiles' split (by 10 to 20 % over gemm.hip's
// kernel where the two are level from HBM): where that is one round, the others have to be 5 % better.
// Whole calls from HBM: gemm.hip's four waves always -> few_tiles' split always -> so chosen: 18944 x 4096 at 64 tokens MLX 4-bit 34.0 us -> 40.7 (296
// workgroups) -> 32.8, Q4_K 38.2 -> 45.6 -> 34.4, at 24 tokens 31.7 -> 33.3 -> 28.2 and 36.0 -> 37.9 -> 30.7 (three row tiles); 128256 x 2048 at 64 MLX
// 4-bit 74.5 -> 103.6 -> 72.3; Q8_0 17408 x 5120 at 64 48.0 -> 63.7 -> 47.1, 7168 x 14336 53.0 -> 60.2 -> 53.6; Q8 with f32 scales 14336 x 4096 at 64
// 35.5 -> 47.8 -> 34.6, 7168 x 18432 62.1 -> 91.0 -> 61.3; FP8 7168 x 18432 at 64 58.7 -> 60.8 -> 55.7.
struct ShortPlan {
    uint32_t rt, slices;
};
struct ShortCost {
    double row, token, both, unit;
};
inline ShortCost short_cost(int fmt) {
    switch (fmt) {
        case FMT_Q8_0: return {0.577, 0.250, 0.02, 0.771};
        case FMT_Q8F: return {0.464, 0.343, 0.02, 0.676};
        case FMT_Q4_K: return {0.384, 0.318, 0.02, 0.819};
        case FMT_Q5_K: return {0.528, 0.320, 0.02, 0.874};
        case FMT_Q6_K: return {0.471, 0.247, 0.02, 0.773};
        case FMT_FP8: return {0.437, 0.247, 0.02, 0.665};
        case FMT_MXFP4: return {0.412, 0.243, 0.02, 0.852};
        case FMT_NVFP4: return {0.974, 0.184, 0.048, 1.828};
        case FMT_Q40: return {0.255, 0.301, 0.02, 0.764};
        default: return {0.311, 0.299, 0.02, 0.733};  // MLX 4-bit
    }
}
constexpr bool short_form(int fmt, uint32_t ntt, uint32_t rt) { return !(fmt == FMT_Q8F && ntt * rt == 16); }  // (would spill: not built)
// gemm_short.hip's forms of at most 128 registers: two workgroups to a CU
constexpr bool short_pairs(int fmt, uint32_t ntt, uint32_t rt) {
    if (rt * ntt != 6) return rt * ntt < 6;
    return fmt != FMT_Q8_0 && fmt != FMT_Q8F && fmt != FMT_Q5_K && !(fmt == FMT_Q6_K && rt == 3);
}
// Few enough row tiles that the CUs have a workgroup each, and no fewer, since the workgroups of a launch request the whole activations
// once each; K slices where rows are long and the row tiles do not fill the CUs, or let a workgroup have more of them.
inline ShortPlan few_tiles(int fmt, uint32_t tiles, uint32_t steps, size_t t) {
    if (tiles <= 128) return {1, steps >= 64 ? (tiles <= 64 ? 4u : 256 / tiles) : 1};
    if (tiles <= 256) return steps * t >= 4000 ? ShortPlan{2, 2} : ShortPlan{1, 1};
    const uint32_t most = fmt == FMT_Q8F && t > 48 ? 3 : 4;
    if (tiles <= 512) return steps >= (tiles <= 340 ? 96 : 128) ? ShortPlan{most, tiles <= 340 ? 3u : 2u} : ShortPlan{2, 1};
    return {tiles <= 768 ? 3u : most, 1};
}
inline ShortPlan short_plan(int fmt, uint32_t n_out, uint32_t n_in, size_t t) {
    const uint32_t tiles = (n_out + 15) / 16, steps = (n_in + 127) / 128, mtiles = (uint32_t)((t + 15) / 16), ntt = mtiles < 2 ? 2 : mtiles;
    const ShortCost c = short_cost(fmt);
    const double mb = (double)n_out * n_in * 1e-6 * (fmt == FMT_Q8F ? 1.13 : fmt == FMT_Q8_0 || fmt == FMT_FP8 ? 1.0 : fmt == FMT_Q6_K ? 0.82 : fmt == FMT_Q5_K ? 0.69 : 0.56);
    const double all = 5.9 + 0.15 * mb;
    const ShortPlan few = few_tiles(fmt, tiles, steps, t);
    ShortPlan best{0, 1};
    double least = all + 0.97 + c.unit * gemm_plan(fmt, n_out, n_in, mtiles).cost + 1.09 * ntt + 0.03 * mb;
    for (uint32_t rt = 1; rt <= 4; rt++) {
        if (!short_form(fmt, ntt, rt)) continue;
        for (uint32_t z = 1; z <= 4 && (z == 1 || steps >= 16 * z); z++) {
            const uint64_t rounds = ((uint64_t)((tiles + rt - 1) / rt) * z + 255) / 256;
            const double held = short_pairs(fmt, ntt, rt) ? (double)(rounds / 2) * 1.8 + (double)(rounds % 2) : (double)rounds;
            const double wave = steps / (8.0 * z);
            double cost = all + held * (0.166 + 0.168 * rt * ntt + wave * (c.row * rt + c.token * ntt + c.both * rt * ntt)) + 0.017 * steps + (z > 1 ? 1.84 + 2.46e-6 * z * t * n_out : 0);
            if (rt == few.rt && z == few.slices && rounds == 1) cost *= 0.95;
            if (cost < least) {
                least = cost;
                best = ShortPlan{rt, z};
            }
        }
    }
    return best;
}

}  // namespace oxhip

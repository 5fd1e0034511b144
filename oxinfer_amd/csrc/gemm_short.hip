// The bf16 GEMM of up to 64 tokens: y[t][n_out] = x[t][n_in] * W^T for every format of gemm.hip, whose weight operands and packed
// activation fragments it shares. At these sizes the product is bound by the weights' way from memory to the matrix cores: the records
// come in (33 MB of a 14336 x 4096 matrix in 4 bits are 6.5 us), and 23 vector instructions turn each lane's eight codes into an operand.
//
// Work split: every wave is on its own from the first request to the end of its sums. A workgroup of eight waves owns RT row tiles; wave v
// takes the K-steps v, v + 8, ... (of its slice), so that a workgroup reads one contiguous window of its tiles' records, turns each
// record into operands in registers and multiplies it with the fragments of all its NTT token tiles: 4 NTT RT matrix instructions a step,
// no barrier, no weight through LDS. The eight sums meet in LDS once, in wave order. (Sharing the operands of 128 rows through LDS, as
// gemm.hip does for more tokens, put two barriers' waits and a trip through LDS into each of the six to sixteen steps that a workgroup
// has here, and needed K slices, and a launch to add them, for almost every matrix.)
// The fragments are requested by every wave that needs them, RT records to a fragment, so RT is as large as keeps the CUs busy: see
// short_plan. A step's registers are refilled where they are used up, the fragments a step ahead, the records two (three: no gain, the
// kernels of four row tiles spill; read-once requests for the records: 10 to 30 % slower, the other side of a line of scales is lost).
//
// Whole calls on the device, packing included, before (gemm.hip's kernel with four waves of one token tile) -> this, at 24 / 43 / 64 tokens:
// MLX 4-bit 4096 x 4096 14.2 / 16.6 / 17.6 -> 9.2 / 11.3 / 12.4 us, 14336 x 4096 24.4 / 25.2 / 25.9 -> 17.0 / 19.0 / 20.3, 4096 x 14336
// 24.0 / 24.6 / 25.1 -> 19.4 / 21.9 / 23.6; Q4_K 15.6 / 17.4 / 19.2 -> 10.3 / 11.7 / 13.2, 27.5 / 27.6 / 29.0 -> 18.9 / 20.5 / 21.9,
// 26.7 / 27.2 / 28.1 -> 21.9 / 23.7 / 25.4; Q6_K 5001 x 4352 at 43 tokens 19.6 -> 14.0; NVFP4 4096 x 4096 23.6 / 25.1 / 26.8 -> 12.5 / 13.2 / 13.9.
#include <algorithm>
#include <type_traits>

#include "gemm_tile.hpp"

namespace oxhip {

namespace {

constexpr int KW = 8;  // waves of a workgroup, which share its K-steps (four: 10 to 20 % slower but for the smallest matrices)

// grid: (groups of RT row tiles, K slices); blockDim 64 KW. With slices, the sums go out as f32 partial rows [slice][t][n_out].
template <int FMT, int NTT, int RT>
__global__ __launch_bounds__(64 * KW, 2) void gemm_short_kernel(WeightView w, const uint4* __restrict__ apk, uint32_t t, uint32_t mtiles, void* __restrict__ yv,
                                                         uint32_t out_bf16, float* __restrict__ partial) {
    extern __shared__ __align__(16) float red[];  // [KW][RT][NTT][64][4]
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nsteps = (w.n_in + 127) / 128, ntiles = row_tiles(w.n_out), kblocks = 4 * nsteps;
    const uint32_t gw = blockIdx.y * KW + wave, stride = KW * gridDim.y;
    const uint32_t cnt = gw < nsteps ? (nsteps - gw + stride - 1) / stride : 0, slast = cnt ? gw + stride * (cnt - 1) : 0;
    const uint8_t* base[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) base[r] = tile_records<FMT>(w, min(blockIdx.x * RT + r, ntiles - 1), lane);
    f32x4 acc[RT][NTT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int tt = 0; tt < NTT; tt++) acc[r][tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto load_w = [&](RawTile* raw, uint32_t s) {
#pragma unroll
        for (int r = 0; r < RT; r++) load_tile<FMT>(raw[r], w, base[r], min(blockIdx.x * RT + r, ntiles - 1), s, lane);
    };
    // (token tiles past the last repeat it; their sums are not stored)
    auto load_a = [&](uint4* a, uint32_t blk) {
#pragma unroll
        for (int tt = 0; tt < NTT; tt++) {
            const uint64_t pa = reinterpret_cast<uint64_t>(apk + ((size_t)min((uint32_t)tt, mtiles - 1) * kblocks + blk) * 64);
            const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)pa), hi = __builtin_amdgcn_readfirstlane((uint32_t)(pa >> 32));
            a[tt] = __builtin_bit_cast(uint4, reinterpret_cast<const __attribute__((address_space(1))) u32x4g*>(((uint64_t)hi << 32) | lo)[lane]);
        }
    };
    constexpr int PF = 2;  // steps of records on request
    RawTile raw[PF][RT];
    uint4 a[4][NTT];
    load_w(raw[0], min(gw, slast));
#pragma unroll
    for (int b = 0; b < 4; b++) load_a(a[b], 4 * min(gw, slast) + b);
#pragma unroll
    for (int p = 1; p < PF; p++) load_w(raw[p], min(gw + p * stride, slast));
    for (uint32_t i = 0; i < cnt; i += PF) {
#pragma unroll
        for (int p = 0; p < PF; p++) {
            const uint32_t s = min(gw + stride * (i + p), slast), s1 = min(s + stride, slast), s2 = min(s + PF * stride, slast);
            if (i + p < cnt) {
#pragma unroll
                for (int b = 0; b < 4; b++) {
#pragma unroll
                    for (int r = 0; r < RT; r++) {
                        const bf16x8 bb = __builtin_bit_cast(bf16x8, tile_block<FMT>(raw[p][r], w, b, s, lane));
#pragma unroll
                        for (int tt = 0; tt < NTT; tt++)
                            acc[r][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[b][tt]), bb, acc[r][tt], 0, 0, 0);
                    }
                    load_a(a[b], 4 * s1 + b);
                }
            }
            load_w(raw[p], s2);
        }
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int tt = 0; tt < NTT; tt++) *reinterpret_cast<f32x4*>(red + ((((size_t)wave * RT + r) * NTT + tt) * 64 + lane) * 4) = acc[r][tt];
    __syncthreads();
    // D[token 4 kq + i][row n]: thread (r, tt, lane) adds the waves in order and stores its four tokens
    for (uint32_t idx = threadIdx.x; idx < RT * NTT * 64; idx += blockDim.x) {
        const uint32_t l = idx & 63, tt = (idx >> 6) % NTT, r = (idx >> 6) / NTT;
        const uint32_t row = (blockIdx.x * RT + r) * 16 + (l & 15);
        if (row >= w.n_out) continue;
        f32x4 sum = *reinterpret_cast<const f32x4*>(red + (((size_t)r * NTT + tt) * 64 + l) * 4);
        for (uint32_t k = 1; k < KW; k++) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(red + ((((size_t)k * RT + r) * NTT + tt) * 64 + l) * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) sum[i] += v[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t tok = 16 * tt + 4 * (l >> 4) + i;
            if (tok >= t) continue;
            if (gridDim.y > 1) partial[((size_t)blockIdx.y * t + tok) * w.n_out + row] = sum[i];
            else if (out_bf16) reinterpret_cast<uint16_t*>(yv)[(size_t)tok * w.n_out + row] = f32_to_bf16_bits(sum[i]);
            else reinterpret_cast<float*>(yv)[(size_t)tok * w.n_out + row] = sum[i];
        }
    }
}

// Row tiles per workgroup and K slices, by measuring 30 shapes from 1024 x 2048 to 14336 x 14336 in up to five formats (device time of
// whole calls, Q4_K at 24 and 64 tokens where nothing else is said): few enough row tiles that the 256 CUs have a workgroup each, and
// no fewer, since the workgroups of a launch request the whole activations once each.
//   4096 x 4096, MLX 4-bit: one row tile 9.8 and 13.1 us, two (128 workgroups) 11.4 and 14.0, four 14.7 and 19.0.
//   5001 x 4352, MLX 4-bit: two (157 workgroups) 12.0 and 14.9, one (313: some CUs have two) 13.9 and 19.9, four 15.5 and 19.0.
//   12000 x 4096: three (250 workgroups) 16.4 and 19.1, two (375) 19.1 and 25.4, four (188) 17.9 and 21.5; 8320 rows 15.4 and 18.9, 17.7
//   and 24.7, 17.4 and 21.3. 14336 x 4096, MLX 4-bit: four (224 workgroups) 17.2 and 20.2, two (448) 17.0 and 23.4, one 21.7 and 30.6.
// K slices cost a launch that adds them. They pay where rows are long and the row tiles do not fill the CUs (1024 x 14336: whole 19.4 and
// 28.4, in four slices 12.9 and 17.4; x 8192 13.6 and 18.4, 10.2 and 13.0; x 4096 9.7 and 12.6, 9.1 and 10.8, which the host's third
// launch takes back), or where they let a workgroup have more row tiles, which halves the fragments' requests:
//   4096 x 14336, MLX 4-bit: one tile, whole 19.3 and 29.2 us (24.3 at 48 tokens), two tiles in two slices 19.1 and 24.9 (22.4).
//   4096 x 11008 at 48 / 64 tokens 19.4 / 24.5, 19.4 / 22.6; 3000 x 8192 at 40 / 64 16.7 / 19.4, 16.8 / 18.5.
//   5120 x 12288: two tiles, whole 27.1 and 31.0, four in three slices (240 workgroups) 21.2 and 25.9; FP8 at 64 28.0 and 25.6.
//   7168 x 18432 at 64: FP8 54.1 and (four, two slices) 47.4, Q8_0 56.9 and 52.0, Q6_K 49.3 and 47.6, MLX 4-bit 38.3 and 37.7.
//   7168 x 14336 is better whole (Q5_K 32.5 and 36.6; 30.9 and 37.6), as are 8192 x 8192 and 14336 rows of 8192 and 14336 columns.
// (Q8 at four token tiles keeps to three row tiles: four would spill.)
struct ShortPlan {
    uint32_t rt, slices;
};
ShortPlan short_plan(const WeightView& w, size_t t) {
    const uint32_t tiles = row_tiles(w.n_out), steps = (w.n_in + 127) / 128;
    if (tiles <= 128) return {1, steps >= 64 ? std::min(4u, 256 / tiles) : 1};
    if (tiles <= 256) return steps * t >= 4000 ? ShortPlan{2, 2} : ShortPlan{1, 1};
    const uint32_t most = w.fmt == FMT_Q8F && t > 48 ? 3 : 4;
    if (tiles <= 512) return steps >= (tiles <= 340 ? 96 : 128) ? ShortPlan{most, tiles <= 340 ? 3u : 2u} : ShortPlan{2, 1};
    return {tiles <= 768 ? 3u : most, 1};
}

}  // namespace

bool gemm_short_ok(size_t t) { return t <= 64; }
uint32_t gemm_short_slices(const WeightView& w, size_t t) { return short_plan(w, t).slices; }

namespace {

template <int FMT>
hipError_t run_short(const WeightView& w, const void* apk, size_t t, void* y, bool out_bf16, float* partial, hipStream_t s) {
    const ShortPlan p = short_plan(w, t);
    const uint32_t mtiles = (uint32_t)((t + 15) / 16);
    hipError_t e = hipSuccess;
    auto go = [&](auto ntt, auto rt) {
        constexpr int NTT = decltype(ntt)::value, RT = decltype(rt)::value;
        if constexpr (!(FMT == FMT_Q8F && NTT * RT == 16)) {
            auto kern = gemm_short_kernel<FMT, NTT, RT>;
            constexpr size_t lds = (size_t)KW * RT * NTT * 1024;
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e == hipSuccess) kern<<<dim3((row_tiles(w.n_out) + RT - 1) / RT, p.slices), 64 * KW, lds, s>>>(w, static_cast<const uint4*>(apk), (uint32_t)t, mtiles, y, out_bf16, partial);
        } else {
            e = hipErrorInvalidValue;  // (short_plan keeps from it)
        }
    };
    auto tokens = [&](auto rt) {
        if (mtiles <= 2) go(std::integral_constant<int, 2>{}, rt);
        else if (mtiles == 3) go(std::integral_constant<int, 3>{}, rt);
        else go(std::integral_constant<int, 4>{}, rt);
    };
    span_start(s);
    if (p.rt == 1) tokens(std::integral_constant<int, 1>{});
    else if (p.rt == 2) tokens(std::integral_constant<int, 2>{});
    else if (p.rt == 3) tokens(std::integral_constant<int, 3>{});
    else tokens(std::integral_constant<int, 4>{});
    if (e == hipSuccess) e = hipGetLastError();
    span_stop(s);
    if (e != hipSuccess || p.slices == 1) return e;
    return launch_gemm_reduce(partial, t * (size_t)w.n_out, p.slices, y, out_bf16, s);
}

}  // namespace

// `apk`: the fragments that launch_pack_a makes in gemm_bf16_pack_mode; `partial`: gemm_short_slices() * t * n_out floats, if more than one.
hipError_t launch_gemm_short(const WeightView& w, const void* apk, size_t t, void* y, bool out_bf16, float* partial, hipStream_t s) {
    switch (w.fmt) {
        case FMT_Q4M: return run_short<FMT_Q4M>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q40: return run_short<FMT_Q40>(w, apk, t, y, out_bf16, partial, s);
        case FMT_MXFP4: return run_short<FMT_MXFP4>(w, apk, t, y, out_bf16, partial, s);
        case FMT_NVFP4: return run_short<FMT_NVFP4>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q8_0: return run_short<FMT_Q8_0>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q8F: return run_short<FMT_Q8F>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q4_K: return run_short<FMT_Q4_K>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q5_K: return run_short<FMT_Q5_K>(w, apk, t, y, out_bf16, partial, s);
        case FMT_Q6_K: return run_short<FMT_Q6_K>(w, apk, t, y, out_bf16, partial, s);
        case FMT_FP8: return run_short<FMT_FP8>(w, apk, t, y, out_bf16, partial, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace oxhip

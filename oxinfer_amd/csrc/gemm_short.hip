// The bf16 GEMM of up to 64 tokens: y[t][n_out] = x[t][n_in] * W^T for every format of gemm.hip, whose weight operands and packed
// activation fragments it shares. At these sizes the product is bound by the weights' way from memory to the matrix cores: the records
// come in (33 MB of a 14336 x 4096 matrix in 4 bits are 6.5 us), and 23 vector instructions turn each lane's eight codes into an operand.
//
// Work split: every wave is on its own from the first request to the end of its sums. A workgroup of eight waves owns RT row tiles; wave v
// takes the K-steps v, v + 8, ... (of its slice), so that a workgroup reads one contiguous window of its tiles' records, turns each
// record into operands in registers and multiplies it with the fragments of all its NTT token tiles: 4 NTT RT matrix instructions a step,
// no barrier, no weight through LDS. The eight sums meet in LDS once, in wave order. (Sharing the operands of 128 rows through LDS, as
// gemm.hip does for more tokens, puts two barriers' waits and a trip through LDS into each of the six to sixteen steps that a workgroup
// has here, and needs K slices, and a launch to add them, for almost every matrix.)
// The fragments are requested by every wave that needs them, RT records to a fragment: row tiles, K slices and the sizes where gemm.hip's
// way is the faster one all the same are short_plan's (gemm_plan.hpp). A step's registers are refilled where they are used up, the fragments
// a step ahead, the records two (three: no gain, the kernels of four row tiles spill; read-once requests for the records: 10 to 30 %
// slower, the other side of a line of scales is lost).
//
// Whole calls on the device, packing included, weights in HBM (in brackets: in the Infinity Cache), gemm.hip's four waves -> this, at 24 / 43 /
// 64 tokens: MLX 4-bit 4096 x 4096 15.3 / 16.6 / 18.2 -> 11.4 / 13.8 / 15.5 us (13.4 / 15.1 / 16.7 -> 8.8 / 10.3 / 12.0), 14336 x 4096 25.8 / 27.2 / 28.6
// -> 21.3 / 23.5 / 25.5 (22.5 / 23.9 / 25.3 -> 15.5 / 17.4 / 19.3); Q4_K 16.9 / 18.2 / 20.2 -> 12.0 / 14.1 / 15.8, 29.6 / 31.0 / 32.0 -> 22.9 / 25.0 / 27.1;
// Q6_K 5001 x 4352 at 43 tokens 21.8 -> 18.3 (18.9 -> 13.2); NVFP4 4096 x 4096 24.2 / 25.5 / 26.9 -> 13.7 / 14.7 / 16.0.
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

template <int FMT>
hipError_t run_short(const WeightView& w, const void* apk, size_t t, const ShortPlan& p, void* y, bool out_bf16, float* partial, hipStream_t s) {
    const uint32_t mtiles = (uint32_t)((t + 15) / 16);
    hipError_t e = hipSuccess;
    auto go = [&](auto ntt, auto rt) {
        constexpr int NTT = decltype(ntt)::value, RT = decltype(rt)::value;
        if constexpr (short_form(FMT, NTT, RT)) {
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

// `apk`: the fragments that launch_pack_a makes in gemm_bf16_pack_mode; `partial`: p.slices * t * n_out floats, if more than one.
hipError_t launch_gemm_short(const WeightView& w, const void* apk, size_t t, const ShortPlan& p, void* y, bool out_bf16, float* partial, hipStream_t s) {
    switch (w.fmt) {
        case FMT_Q4M: return run_short<FMT_Q4M>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q40: return run_short<FMT_Q40>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_MXFP4: return run_short<FMT_MXFP4>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_NVFP4: return run_short<FMT_NVFP4>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q8_0: return run_short<FMT_Q8_0>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q8F: return run_short<FMT_Q8F>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q4_K: return run_short<FMT_Q4_K>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q5_K: return run_short<FMT_Q5_K>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_Q6_K: return run_short<FMT_Q6_K>(w, apk, t, p, y, out_bf16, partial, s);
        case FMT_FP8: return run_short<FMT_FP8>(w, apk, t, p, y, out_bf16, partial, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace oxhip

// quantize_act (src/quant.rs:267-292 of the reference) of one block of 32 by eight lanes: shared by the stand-alone kernels,
// the fused RMSNorm and the MoE kernels.
#pragma once
#include "internal.hpp"

namespace oxhip {

// The QAct planes a quantization writes.
struct QActOut {
    int8_t* __restrict__ q;
    float* __restrict__ scales;
    int32_t* __restrict__ sums;
    float* __restrict__ fsums;
    float* __restrict__ hsums;
    int32_t* __restrict__ sums16;
};
inline QActOut qact_out(const oxhip_qact& o) { return QActOut{o.q, o.scales, o.sums, o.fsums, o.hsums, o.sums16}; }

template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

// One block of 32 by the eight lanes 8 g .. 8 g + 7 of a wave, all of them here together: lane `part` = 0..7 brings elements
// 4 part .. 4 part + 3 in `v`; the block is number b of the output arrays. Every output is the reference's bit for bit. The
// maximum, the codes and the integer sums do not depend on the order; the f32 sums do and are formed in element order, the
// running sum handed from lane to lane (Rust's iter().sum() starts from -0.0: an all -0.0 block sums to -0.0).
// These kernels are single waves' latency: one lane walking a whole block was some 500 instructions at five to eight cycles
// each, the eight lanes take about 120 and read whole lines (quantize_act of 4096 values 3.9 -> 3.6 us, RMSNorm and
// quantization 5.4 -> 4.4 us, in a replayed chain, launch boundary included; on an idle stream 3.05 -> 2.35 us).
__device__ __forceinline__ void quantize_act_part(const float* v, uint32_t part, size_t b, const QActOut& o) {
    // (from zero, as the reference: the maximum passes NaNs over, and a block of nothing else has the scale 0)
    float amax = fmaxf(fmaxf(fmaxf(0.0f, fabsf(v[0])), fabsf(v[1])), fmaxf(fmaxf(0.0f, fabsf(v[2])), fabsf(v[3])));
    amax = fmaxf(amax, dpp_f32<0xB1>(amax));   // quad_perm [1,0,3,2]
    amax = fmaxf(amax, dpp_f32<0x4E>(amax));   // quad_perm [2,3,0,1]
    amax = fmaxf(amax, dpp_f32<0x141>(amax));  // row_half_mirror: the other four lanes
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
    uint32_t packed = 0;
    int s = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float r = roundf(v[i] * inv);  // half away from zero
        const int iv = r != r ? 0 : (int)fminf(fmaxf(r, -128.0f), 127.0f);
        s += iv;
        packed |= ((uint32_t)iv & 0xFF) << (8 * i);
    }
    s += dpp_i32<0xB1>(s);
    s += dpp_i32<0x4E>(s);  // the half's sum, in its four lanes
    const int s_all = s + dpp_i32<0x141>(s);
    // the halves: lane 4 h starts from -0.0, its right neighbour goes on from its sum, ...; lanes 3 and 7 end with h0 and h1
    float h = -0.0f;
#pragma unroll
    for (int step = 0; step < 4; step++) {
        const float in = dpp_f32<0x111>(h);  // row_shr:1
        h = (part & 3) == 0 ? -0.0f : in;
        h = ((h + v[0]) + v[1]) + v[2];
        h = h + v[3];
    }
    // the block: lane 4 goes on from h0
    float f = h;
#pragma unroll
    for (int step = 0; step < 4; step++) {
        const float in = dpp_f32<0x111>(f);
        const float g = (((in + v[0]) + v[1]) + v[2]) + v[3];
        f = part < 4 ? f : g;
    }
    *reinterpret_cast<uint32_t*>(o.q + b * 32 + 4 * part) = packed;
    if (part == 3) {
        o.scales[b] = amax / 127.0f;
        o.hsums[2 * b] = h;
        o.sums16[2 * b] = s;
    } else if (part == 7) {
        o.sums[b] = s_all;
        o.fsums[b] = f;
        o.hsums[2 * b + 1] = h;
        o.sums16[2 * b + 1] = s;
    }
}

// Blocks of 32 of x, eight lanes each: lane i of the launch's lanes takes part i % 8 of block i / 8.
__device__ __forceinline__ void quantize_act_lane(const float* __restrict__ x, size_t i, size_t nblocks, const QActOut& o) {
    const size_t b = i >> 3;
    if (b >= nblocks) return;  // (uniform over a block's eight lanes)
    const float4 f = *reinterpret_cast<const float4*>(x + 4 * i);
    const float v[4] = {f.x, f.y, f.z, f.w};
    quantize_act_part(v, (uint32_t)i & 7, b, o);
}

// fast_exp of the reference (src/kernels.rs:2225-2231): clamp, Cody-Waite reduction, degree-6 polynomial,
// scale by 2^fx through the exponent bits; every operation unfused as written there.
__device__ __forceinline__ float fast_exp(float x) {
    x = fminf(fmaxf(x, -87.0f), 88.0f);
    const float fx = roundf(x * 1.44269504088896340736f);
    const float r = (x - fx * 0.693359375f) - fx * -2.12194440e-4f;
    const float p = 1.0f + r * (1.0f + r * (0.5f + r * (0.16666667f + r * (0.041666668f + r * (0.008333334f + r * 0.0013888889f)))));
    return __int_as_float(((int)fx + 127) << 23) * p;
}

// Act::apply of one pair (src/moe.rs:18-37, silu_mul / gelu_mul): kind 0 SiLU, 1 GELU-tanh, 2 SiLU with clamp `param`.
__device__ __forceinline__ float gated_act(float g, float u, uint32_t kind, float param) {
    if (kind == 1) {
        const float K2 = 2.0f * 0.7978846f;
        const float t = K2 * (g + 0.044715f * g * g * g);
        return g / (1.0f + fast_exp(-t)) * u;
    }
    if (kind == 2) {
        g = fminf(g, param);
        u = fminf(fmaxf(u, -param), param);
    }
    return g / (1.0f + fast_exp(-g)) * u;
}

// Act::scalar (src/moe.rs:39-46), what the reference's grouped prefill path applies: the exponential of the SiLU
// kinds is the library's, not fast_exp (GELU-tanh goes through fast_exp in both, src/kernels.rs:2235-2239).
__device__ __forceinline__ float gated_act_scalar(float g, float u, uint32_t kind, float param) {
    if (kind == 1) return gated_act(g, u, kind, param);
    if (kind == 2) {
        g = fminf(g, param);
        u = fminf(fmaxf(u, -param), param);
    }
    return g / (1.0f + expf(-g)) * u;
}

}  // namespace oxhip

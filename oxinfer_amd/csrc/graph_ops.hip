// Kernels of the single-token decode graph around the matmuls (the reference's Op list, src/gpu_decode.rs:52-340):
// the output modes of a linear for the formats whose decode kernels only store, the gate / up pair as an elementwise
// op (Op::Glu), the router's logits (Op::Route before its top-k), and RMSNorm fused with the activation quantization
// that the next matmul reads (Op::Norm feeding Op::Linear; rmsnorm, src/kernels.rs:2107-2123, then quantize_act,
// src/quant.rs:243-343).
#include "act_body.hpp"
#include "internal.hpp"

namespace oxhip {

__global__ __launch_bounds__(256) void epilogue_kernel(const float* __restrict__ v, uint32_t n, size_t total, float* __restrict__ y, Epi epi) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const float x = v[i];
    if (epi.mode == EPI_STORE) y[i] = x;
    else if (epi.mode == EPI_ADD) y[i] = y[i] + x;
    else y[i] = y[i] + (1.0f / (1.0f + expf(-epi.gate[i / n]))) * x;
}

hipError_t launch_epilogue(const float* v, size_t t, size_t n, float* y, const Epi& epi, hipStream_t s) {
    const size_t total = t * n;
    if (!total) return hipSuccess;
    epilogue_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(v, (uint32_t)n, total, y, epi);
    return hipGetLastError();
}

// y = silu(g) * u or gelu_tanh(g) * u (silu_mul / gelu_mul, src/kernels.rs:2188-2198, :2234-2257: both through fast_exp).
__global__ __launch_bounds__(256) void glu_kernel(const float* __restrict__ g, const float* __restrict__ u, size_t n, uint32_t kind,
                                                  float* __restrict__ y) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = gated_act(g[i], u[i], kind, 0.0f);
}

hipError_t launch_glu(const float* g, const float* u, size_t n, bool gelu, float* y, hipStream_t s) {
    if (!n) return hipSuccess;
    glu_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(g, u, n, gelu ? 1u : 0u, y);
    return hipGetLastError();
}

// logits[tok][e] = router[e] . x[tok] for e < n_exp, and with `gate` one more logit gate . x[tok] behind them
// (Op::Route, src/gpu_decode.rs:154-172). One wavefront per logit: f32 rows read as whole lines, f32 accumulation.
__global__ __launch_bounds__(512) void router_logits_kernel(const float* __restrict__ x, const float* __restrict__ router,
                                                            const float* __restrict__ gate, uint32_t n_exp, uint32_t h,
                                                            float* __restrict__ logits) {
    const uint32_t lane = threadIdx.x & 63, row = blockIdx.x * 8 + (threadIdx.x >> 6), tok = blockIdx.y;
    const uint32_t rows = n_exp + (gate ? 1u : 0u);
    if (row >= rows) return;
    const float* w = row < n_exp ? router + (size_t)row * h : gate;
    const float* xr = x + (size_t)tok * h;
    float acc = 0.0f;
    if (h % 4 == 0) {
        for (uint32_t i = 4 * lane; i < h; i += 256) {
            const float4 a = *reinterpret_cast<const float4*>(w + i), b = *reinterpret_cast<const float4*>(xr + i);
            acc = fmaf(a.x, b.x, acc);
            acc = fmaf(a.y, b.y, acc);
            acc = fmaf(a.z, b.z, acc);
            acc = fmaf(a.w, b.w, acc);
        }
    } else {
        for (uint32_t i = lane; i < h; i += 64) acc = fmaf(w[i], xr[i], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) logits[(size_t)tok * rows + row] = acc;
}

hipError_t launch_router_logits(const float* x, const float* router, const float* gate, size_t t, size_t n_exp, size_t h, float* logits,
                                hipStream_t s) {
    const size_t rows = n_exp + (gate ? 1 : 0);
    if (!t || !rows) return hipSuccess;
    router_logits_kernel<<<dim3((unsigned)((rows + 7) / 8), (unsigned)t), 512, 0, s>>>(x, router, gate, (uint32_t)n_exp, (uint32_t)h, logits);
    return hipGetLastError();
}

// The correctly rounded f32 of m^(-1/2), m = ss / n + eps: in f64, from the hardware's estimate by two Newton steps, which round
// to the f32 of 1 / sqrt(m) for every float of the range that takes them (compared over all 2.0e9), and as that quotient outside
// it. The quotient and the root alone are some 50 dependent f64 instructions.
__device__ __forceinline__ float rms_factor(double ss, uint32_t n, float eps) {
    const float m = (float)ss / (float)n + eps;
    const double d = (double)m;
    if (!(m >= 0x1p-120f && m <= 0x1p120f)) return (float)(1.0 / sqrt(d));
    double y = __builtin_amdgcn_rsq(d);
#pragma unroll
    for (int i = 0; i < 2; i++) y = fma(y, 0.5 * fma(-d * y, y, 1.0), y);
    return (float)y;
}

// The sum over a wave's 64 lanes, in every lane: lanes 32 apart first, then 16, 8, 4, 2 and 1 (a fixed order). In registers: the
// halves and quarters change places with the lane swaps; from 8 on the values repeat, so that rotations within 16 lanes bring them.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, ((uint64_t)(uint32_t)dpp_i32<CTRL>((int)(b >> 32)) << 32) | (uint32_t)dpp_i32<CTRL>((int)(uint32_t)b));
}
__device__ __forceinline__ double wave_xor_sum(double v) {
    auto swap_add = [](double a, auto swap) {
        const uint64_t b = __builtin_bit_cast(uint64_t, a);
        const auto lo = swap((uint32_t)b), hi = swap((uint32_t)(b >> 32));
        return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) + __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
    };
    v = swap_add(v, [](uint32_t x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
    v = swap_add(v, [](uint32_t x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    v += dpp_f64<0x128>(v);  // row_ror:8
    v += dpp_f64<0x124>(v);  // row_ror:4
    v += dpp_f64<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_f64<0xB1>(v);   // quad_perm [1,0,3,2]
    return v;
}

// RMSNorm of one row per workgroup (Op::Norm, src/gpu_decode.rs:53-66), then quantize_act of the row that was written,
// without a round trip through memory:
//   x' = x * pre;  r = (sum x'^2 / n + eps)^(-1/2);  v = (x' * r) * w  (or x' * r);  out = v, or out += v with `add`;
//   what `out` then holds goes, per block of 32, to the QAct (optional).
// The reference sums the squares one after the other in f32 (src/kernels.rs:2109), which no parallel machine can
// repeat bit for bit in useful time: here the squares are exact in f64 and summed in f64 (a fixed order), the mean and
// eps added in f32 as the reference does, and r is the correctly rounded power. The quantization of v is
// quantize_act's, bit for bit (the same code on the same values). VEC: rows of x, out and w start on 16-byte boundaries
// (float4 access); otherwise every access is one float.
// The kernel is one row's chain of latencies, so a row takes as many threads as it has float4s (up to 1024), its values and
// weights are requested together and stay in registers (NV float4s a thread; NV = 0: longer rows, read twice), and eight
// lanes quantize a block where they hold it (4096 values, one row, in a replayed chain: 5.4 -> 4.4 us).
// ONE row in one workgroup: rows that share memory with an output, very long rows, and launches of so many rows that they fill
// the chip; the others go to rmsnorm_parts_kernel below, value for value.
template <bool VEC, int NV>
__global__ __launch_bounds__(1024) void rmsnorm_quantize_kernel(const float* __restrict__ x, const float* __restrict__ w_f32,
                                                                const uint16_t* __restrict__ w_bf16, float eps, float pre, uint32_t add, uint32_t n,
                                                                size_t x_stride, size_t out_stride, float* __restrict__ out, QActOut q) {
    __shared__ double part_s[16];
    const uint32_t tok = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nthr = blockDim.x, nwaves = nthr >> 6;
    const float* xr = x + (size_t)tok * x_stride;
    auto load4 = [&](const float* p, float* v) {
        if constexpr (VEC) {
            const float4 f = *reinterpret_cast<const float4*>(p);
            v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        } else {
            v[0] = p[0]; v[1] = p[1]; v[2] = p[2]; v[3] = p[3];
        }
    };
    auto load_w = [&](uint32_t i, float* v) {
        if (w_f32) {
            load4(w_f32 + i, v);
        } else if (w_bf16) {
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = bf16_bits_to_f32(w_bf16[i + j]);
        } else {
            v[0] = v[1] = v[2] = v[3] = 1.0f;  // (x * 1 is x)
        }
    };
    float xv[NV ? NV : 1][4], wv[NV ? NV : 1][4];
    double ss = 0.0;
    auto square = [&](const float* v) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float p = v[j] * pre;
            ss += (double)p * p;
        }
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const uint32_t i = 4 * (threadIdx.x + k * nthr);
            if (i < n) {
                load4(xr + i, xv[k]);
                load_w(i, wv[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (4 * (threadIdx.x + k * nthr) < n) square(xv[k]);
    } else {
        for (uint32_t i = 4 * threadIdx.x; i < n; i += 4 * nthr) {
            load4(xr + i, xv[0]);
            square(xv[0]);
        }
    }
    ss = wave_xor_sum(ss);
    if (lane == 0) part_s[wave] = ss;
    __syncthreads();
    double p[16];  // (all requested at once, added in pairs)
#pragma unroll
    for (int i = 0; i < 16; i++) p[i] = part_s[i];
#pragma unroll
    for (int i = 0; i < 16; i++) p[i] = (uint32_t)i < nwaves ? p[i] : 0.0;
#pragma unroll
    for (int d = 1; d < 16; d *= 2)
#pragma unroll
        for (int i = 0; i + d < 16; i += 2 * d) p[i] += p[i + d];
    const float r = rms_factor(p[0], n, eps);
    auto finish = [&](uint32_t i, const float* xs, const float* ws) {  // elements i .. i + 3 of the row
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = ((xs[j] * pre) * r) * ws[j];
        if (out) {
            float* o = out + (size_t)tok * out_stride + i;
            if (add) {
                float f[4];
                load4(o, f);
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = f[j] + v[j];
            }
            if constexpr (VEC) {
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) o[j] = v[j];
            }
        }
        if (q.q) quantize_act_part(v, (i >> 2) & 7, (size_t)tok * (n / 32) + i / 32, q);
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const uint32_t i = 4 * (threadIdx.x + k * nthr);
            if (i < n) finish(i, xv[k], wv[k]);
        }
    } else {
        for (uint32_t i = 4 * threadIdx.x; i < n; i += 4 * nthr) {
            load4(xr + i, xv[0]);
            load_w(i, wv[0]);
            finish(i, xv[0], wv[0]);
        }
    }
}

// The same for few rows, each over several workgroups: a row alone kept one CU busy for 16 waves' worth of instructions while the
// others idled. Every workgroup of a row reads the whole row for the sum of squares (from L2; four waves, one per SIMD, each
// in the place of four waves of the kernel above, so that the sum is the same to the bit) and finishes 1024 values of it.
// In a replayed chain, launch boundary included: 4096 values 3.9 -> 2.55 us, 16 rows 4.25 -> 2.8; 14336 values 7.1 -> 3.6.
// NV as above (1 to 4 float4s per thread of the kernel above, so 4 to 16 here). No output may share memory with the input.
template <bool VEC, int NV>
__global__ __launch_bounds__(256) void rmsnorm_parts_kernel(const float* __restrict__ x, const float* __restrict__ w_f32, const uint16_t* __restrict__ w_bf16,
                                                            float eps, float pre, uint32_t add, uint32_t n, size_t x_stride, size_t out_stride,
                                                            float* __restrict__ out, QActOut q) {
    __shared__ double part_s[16];
    const uint32_t tok = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nthr = n >= 4096 ? 1024u : (n / 4 + 63) / 64 * 64;  // threads of a row in the kernel above
    const float* xr = x + (size_t)tok * x_stride;
    auto load4 = [&](const float* p, float* v) {
        if constexpr (VEC) {
            const float4 f = *reinterpret_cast<const float4*>(p);
            v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        } else {
            v[0] = p[0]; v[1] = p[1]; v[2] = p[2]; v[3] = p[3];
        }
    };
    // everything is requested at once: the row (clamped: no request under a condition), the thread's own four values and weights
    const uint32_t own = 4 * (blockIdx.x * 256 + threadIdx.x), at = min(own, n - 4);
    float xv[4][NV][4], xo[4], wo[4] = {1.0f, 1.0f, 1.0f, 1.0f}, f[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int k = 0; k < NV; k++) load4(xr + min(4 * (64 * (wave + 4 * j) + lane + k * nthr), n - 4), xv[j][k]);
    load4(xr + at, xo);
    if (w_f32) {
        load4(w_f32 + at, wo);
    } else if (w_bf16) {
#pragma unroll
        for (int i = 0; i < 4; i++) wo[i] = bf16_bits_to_f32(w_bf16[at + i]);
    }
    float* o = out ? out + (size_t)tok * out_stride + at : nullptr;
    if (add) load4(o, f);
    double ss[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        ss[j] = 0.0;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const bool live = 64 * (wave + 4 * j) < nthr && 4 * (64 * (wave + 4 * j) + lane + k * nthr) < n;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float p = xv[j][k][i] * pre;
                ss[j] += live ? (double)p * p : 0.0;
            }
        }
        ss[j] = wave_xor_sum(ss[j]);
    }
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) part_s[wave + 4 * j] = ss[j];
    }
    __syncthreads();
    double p[16];
#pragma unroll
    for (int i = 0; i < 16; i++) p[i] = part_s[i];
#pragma unroll
    for (int d = 1; d < 16; d *= 2)
#pragma unroll
        for (int i = 0; i + d < 16; i += 2 * d) p[i] += p[i + d];
    const float r = rms_factor(p[0], n, eps);
    if (own >= n) return;  // (whole blocks of 32: n is a multiple of 32)
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = ((xo[i] * pre) * r) * wo[i];
    if (out) {
        if (add) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = f[i] + v[i];
        }
        if constexpr (VEC) {
            *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = v[i];
        }
    }
    if (q.q) quantize_act_part(v, (own >> 2) & 7, (size_t)tok * (n / 32) + own / 32, q);
}

hipError_t launch_rmsnorm_quantize(const float* x, const float* w_f32, const uint16_t* w_bf16, float eps, size_t t, size_t n, float* out,
                                   const oxhip_qact* qa, hipStream_t s, float pre, bool add, size_t x_stride, size_t out_stride) {
    if (!t || !n) return hipSuccess;
    if (n % 32) return hipErrorInvalidValue;
    if (!x_stride) x_stride = n;
    if (!out_stride) out_stride = n;
    auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const bool vec = al(x) && al(out) && al(w_f32) && x_stride % 4 == 0 && out_stride % 4 == 0;
    const unsigned threads = (unsigned)(n / 4 >= 1024 ? 1024 : (n / 4 + 63) / 64 * 64);
    auto go = [&](auto kern) {
        kern<<<(unsigned)t, threads, 0, s>>>(x, w_f32, w_bf16, eps, pre, add ? 1u : 0u, (uint32_t)n, x_stride, out_stride, out, qa ? qact_out(*qa) : QActOut{});
    };
    // Few rows, several workgroups each (see rmsnorm_parts_kernel): up to two such workgroups per CU, where both were measured (512 of
    // them, 128 rows of 4096: 4.45 -> 3.4 us; 448, 64 rows of 8192: 5.8 -> 3.9). A row that an output shares memory with must have
    // been read before anything is written.
    const unsigned parts = (unsigned)((n + 1023) / 1024);
    auto addr = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
    auto apart = [&](const void* p, size_t bytes) {  // an output from the rows and the weights
        auto from = [&](const void* in, size_t len) { return !p || !in || addr(p) >= addr(in) + len || addr(p) + bytes <= addr(in); };
        return from(x, ((t - 1) * x_stride + n) * 4) && from(w_f32, n * 4) && from(w_bf16, n * 2);
    };
    const size_t nb = t * n / 32;
    if (parts > 1 && n <= 16384 && t * parts <= 512 && apart(out, ((t - 1) * out_stride + n) * 4) &&
        (!qa || (apart(qa->q, nb * 32) && apart(qa->scales, nb * 4) && apart(qa->sums, nb * 4) && apart(qa->fsums, nb * 4) && apart(qa->hsums, nb * 8) && apart(qa->sums16, nb * 8)))) {
        auto go_parts = [&](auto kern) {
            kern<<<dim3(parts, (unsigned)t), 256, 0, s>>>(x, w_f32, w_bf16, eps, pre, add ? 1u : 0u, (uint32_t)n, x_stride, out_stride, out, qa ? qact_out(*qa) : QActOut{});
        };
        if (n <= 4096) vec ? go_parts(rmsnorm_parts_kernel<true, 1>) : go_parts(rmsnorm_parts_kernel<false, 1>);
        else if (n <= 8192) vec ? go_parts(rmsnorm_parts_kernel<true, 2>) : go_parts(rmsnorm_parts_kernel<false, 2>);
        else vec ? go_parts(rmsnorm_parts_kernel<true, 4>) : go_parts(rmsnorm_parts_kernel<false, 4>);
        return hipGetLastError();
    }
    if (n <= 4096) vec ? go(rmsnorm_quantize_kernel<true, 1>) : go(rmsnorm_quantize_kernel<false, 1>);
    else if (n <= 16384) vec ? go(rmsnorm_quantize_kernel<true, 4>) : go(rmsnorm_quantize_kernel<false, 4>);
    else vec ? go(rmsnorm_quantize_kernel<true, 0>) : go(rmsnorm_quantize_kernel<false, 0>);
    return hipGetLastError();
}

}  // namespace oxhip

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
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
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
    const float m = (float)p[0] / (float)n + eps;
    const float r = (float)(1.0 / sqrt((double)m));
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
    if (n <= 4096) vec ? go(rmsnorm_quantize_kernel<true, 1>) : go(rmsnorm_quantize_kernel<false, 1>);
    else if (n <= 16384) vec ? go(rmsnorm_quantize_kernel<true, 4>) : go(rmsnorm_quantize_kernel<false, 4>);
    else vec ? go(rmsnorm_quantize_kernel<true, 0>) : go(rmsnorm_quantize_kernel<false, 0>);
    return hipGetLastError();
}

}  // namespace oxhip

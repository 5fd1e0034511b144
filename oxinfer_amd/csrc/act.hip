// Activation quantization on the device: quant::quantize_act (src/quant.rs:243-343 of the reference).
//
// Per block of 32: amax = max |x|, inv = 127 / amax (0 for an all-zero block),
// q = round-half-away(x * inv) as int8, scale = amax / 127, the integer block sum, and the f32 sums
// of the block and of each half in element order; every output is bit-identical to the CPU's.
// Eight lanes share a block (act_body.hpp). The work is a few hundred KB at most; it is latency, not bandwidth, that matters here.
#include "act_body.hpp"
#include "internal.hpp"

namespace oxhip {

constexpr unsigned QUANT_THREADS = 256;

__global__ __launch_bounds__(QUANT_THREADS) void quantize_act_kernel(const float* __restrict__ x, size_t nblocks, QActOut o) {
    quantize_act_lane(x, (size_t)blockIdx.x * QUANT_THREADS + threadIdx.x, nblocks, o);
}

// Several activation matrices in one launch (a decode step quantizes the input of every group of matmuls; each launch
// is a few microseconds of latency whatever its size).
struct QuantBatchArgs {
    uint32_t njobs;
    uint32_t first[QUANT_BATCH_MAX + 1];  // first block of 32 of job j; first[njobs] = total
    const float* x[QUANT_BATCH_MAX];
    QActOut o[QUANT_BATCH_MAX];
};

__global__ __launch_bounds__(QUANT_THREADS) void quantize_act_batch_kernel(QuantBatchArgs a) {
    const size_t i = (size_t)blockIdx.x * QUANT_THREADS + threadIdx.x;
    const uint32_t b = (uint32_t)(i >> 3);
    if (b >= a.first[a.njobs]) return;
    uint32_t j = 0;
    while (j + 1 < a.njobs && b >= a.first[j + 1]) j++;
    quantize_act_lane(a.x[j], i - 8 * (size_t)a.first[j], (size_t)(a.first[j + 1] - a.first[j]), a.o[j]);
}

hipError_t launch_quantize_act_batch(const float* const* x, const size_t* t, const size_t* n_in, const oxhip_qact* o, size_t n, hipStream_t s) {
    for (size_t i0 = 0; i0 < n; i0 += QUANT_BATCH_MAX) {
        QuantBatchArgs a{};
        a.njobs = (uint32_t)(n - i0 < (size_t)QUANT_BATCH_MAX ? n - i0 : (size_t)QUANT_BATCH_MAX);
        uint32_t total = 0;
        for (uint32_t j = 0; j < a.njobs; j++) {
            const size_t nb = t[i0 + j] * n_in[i0 + j] / 32;
            if (total + nb > 0x7FFFFFFFu) return hipErrorInvalidValue;
            a.first[j] = total;
            total += (uint32_t)nb;
            a.x[j] = x[i0 + j];
            a.o[j] = qact_out(o[i0 + j]);
        }
        a.first[a.njobs] = total;
        if (!total) continue;
        quantize_act_batch_kernel<<<(unsigned)(((size_t)total * 8 + QUANT_THREADS - 1) / QUANT_THREADS), QUANT_THREADS, 0, s>>>(a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_quantize_act(const float* x, size_t t, size_t n_in, const oxhip_qact& o, hipStream_t s) {
    size_t nblocks = t * n_in / 32;
    if (nblocks == 0) return hipSuccess;
    quantize_act_kernel<<<(unsigned)((nblocks * 8 + QUANT_THREADS - 1) / QUANT_THREADS), QUANT_THREADS, 0, s>>>(x, nblocks, qact_out(o));
    return hipGetLastError();
}

}  // namespace oxhip

// Prefill GEMM, variant (a): weights dequantized to bf16 on the way to the matrix cores, bf16 MFMA with f32
// accumulation. y[t][n_out] = x[t][n_in] * W^T for the tile-packed MLX 4-bit, Q8_0 / Q8, Q4_K and Q6_K formats (and
// FP8 bytes with block scales).
//
// The CPU computes this product from the f32-dequantized rows with one fused multiply-add chain per output
// (matmul_quant_block_prefill + gemm_8x8, src/kernels.rs:1998-2038, src/kernels_x86.rs:296-324 of the reference);
// here weights and activations are rounded to bf16 first, so results agree to bf16 precision, not bit for bit.
//
// Work split: a workgroup of 8 waves (two per SIMD) owns 256 tokens x 128 weight rows; wave v owns the token tiles v
// and v + 8 of the workgroup's sixteen and all 128 rows (2 x 8 MFMA tiles of 16 x 16, 64 accumulator registers). One
// wave per SIMD issues a matrix instruction about every 30 cycles with this loop's vector, LDS and memory
// instructions between them; a second wave fills the pipe while the first dequantizes, provided the two do not
// dequantize at the same time: the waves 0-3 do so in a step's first block, the waves 4-7 in its second. Sharing the
// token dimension keeps the activation requests at one per fragment and workgroup (sharing the rows instead would
// request every fragment twice and run into the vector memory path's 64 bytes per cycle and CU). A
// launch of 65 to 128 tokens runs one tile per wave (34 -> 27 us on the Llama-8B MLP shapes against two), one of at most 64 four waves
// of one tile (64 tokens x 128 rows per workgroup) where gemm_short.hip's kernel would take longer (short_plan).
//   B (weights): each K-step of 128 the waves dequantize the step's 8 row tiles (one each; two each with 4 waves) from the packed
//     records into bf16 MFMA fragments in LDS (double-buffered, one barrier per step); every wave then reads all
//     8 x 4 fragments with ds_read_b128. A weight is dequantized once per workgroup: (code - 8) * d + offset in
//     f32 as one fma(code, d, offset - 8 d), rounded to bf16. The GGUF formats likewise, from their own records:
//     Q8_0 q * d, Q4_K (d * sc) * nibble - dmin * mn, Q6_K (d * sc) * (code - 32) (dequantize_row, src/ggml.rs:707-793
//     of the reference), each as one fma over the unsigned code.
//   A (activations): packed beforehand (pack_a_kernel) into MFMA fragments, one 1 KiB record per (16 tokens,
//     block of 32) in the K order the weight fragments use, so a wave fetches its fragment with one coalesced
//     16-byte-per-lane load straight from global memory / L2, a block ahead of its use.
#include <type_traits>

#include "gemm_tile.hpp"

namespace oxhip {

// Activations [t][n_in] (f32 or bf16) -> fragments [mtile][block][lane][8 bf16]; lane = 16 kq + m holds token
// 16 mtile + m at K positions 32 b + 4 kq + {0..3} then 32 b + 16 + 4 kq + {0..3} (SPLIT, the order of the
// nibble pairs of Q4 bytes) or 32 b + 8 kq + {0..7}. Tokens past t and columns past n_in are zero.
// MODE 2 (FP8 weights read 32 row bytes per lane): block kb = 4 s + b of step s holds columns 128 s + 32 kq + 8 b + j.
// MODE 3 (Q6_K records: a lane owns 16 consecutive columns of each half step): block kb = 4 s + 2 h + e holds columns
// 128 s + 64 h + 16 kq + 8 e + j.
template <int MODE, bool SRC_BF16>
__global__ __launch_bounds__(256) void pack_a_kernel(const void* __restrict__ x, uint32_t t, uint32_t n_in, uint32_t mtiles,
                                                     uint32_t kblocks, uint4* __restrict__ out) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)mtiles * kblocks * 64) return;
    const uint32_t lane = idx & 63, m = lane & 15, kq = lane >> 4;
    const uint32_t b = (idx >> 6) % kblocks, mt = (idx >> 6) / kblocks;
    const uint32_t tok = mt * 16 + m;
    uint32_t pk[4] = {0, 0, 0, 0};
    if (tok < t) {
        // the lane's 8 values are two runs of 4 consecutive columns (SPLIT) or one run of 8: whole runs are fetched with
        // one 8- or 16-byte request each (rows are multiples of 8 columns here), a ragged tail value by value
        const uint32_t k0 = MODE == 1   ? 32 * b + 4 * kq
                            : MODE == 2 ? 128 * (b >> 2) + 32 * kq + 8 * (b & 3)
                            : MODE == 3 ? 128 * (b >> 2) + 64 * ((b >> 1) & 1) + 16 * kq + 8 * (b & 1)
                                        : 32 * b + 8 * kq;
        const uint32_t k1 = MODE == 1 ? k0 + 16 : k0 + 4;  // first column of the second run of 4
        const size_t row = (size_t)tok * n_in;
        if (k1 + 4 <= n_in && n_in % 8 == 0) {
            if (SRC_BF16) {
                const uint16_t* xs = reinterpret_cast<const uint16_t*>(x) + row;
                const uint2 a = *reinterpret_cast<const uint2*>(xs + k0), c = *reinterpret_cast<const uint2*>(xs + k1);
                pk[0] = a.x;
                pk[1] = a.y;
                pk[2] = c.x;
                pk[3] = c.y;
            } else {
                const float* xs = reinterpret_cast<const float*>(x) + row;
                const float4 a = *reinterpret_cast<const float4*>(xs + k0), c = *reinterpret_cast<const float4*>(xs + k1);
                pk[0] = f32_to_bf16_bits(a.x) | ((uint32_t)f32_to_bf16_bits(a.y) << 16);
                pk[1] = f32_to_bf16_bits(a.z) | ((uint32_t)f32_to_bf16_bits(a.w) << 16);
                pk[2] = f32_to_bf16_bits(c.x) | ((uint32_t)f32_to_bf16_bits(c.y) << 16);
                pk[3] = f32_to_bf16_bits(c.z) | ((uint32_t)f32_to_bf16_bits(c.w) << 16);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t k = (j < 4 ? k0 : k1 - 4) + j;
                uint16_t h = 0;
                if (k < n_in) {
                    if (SRC_BF16) h = reinterpret_cast<const uint16_t*>(x)[row + k];
                    else h = f32_to_bf16_bits(reinterpret_cast<const float*>(x)[row + k]);
                }
                pk[j >> 1] |= (uint32_t)h << (16 * (j & 1));
            }
        }
    }
    out[idx] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
}

hipError_t launch_pack_a(const void* x, bool src_bf16, int mode, size_t t, size_t n_in, size_t mtiles, size_t kblocks, void* out,
                         hipStream_t s) {
    size_t total = mtiles * kblocks * 64;
    if (!total) return hipSuccess;
    unsigned grid = (unsigned)((total + 255) / 256);
    uint4* o = static_cast<uint4*>(out);
    const uint32_t tt = (uint32_t)t, kk = (uint32_t)n_in, mt = (uint32_t)mtiles, kb = (uint32_t)kblocks;
    if (mode == 1) {
        if (src_bf16) pack_a_kernel<1, true><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
        else pack_a_kernel<1, false><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
    } else if (mode == 2) {
        if (src_bf16) pack_a_kernel<2, true><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
        else pack_a_kernel<2, false><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
    } else if (mode == 3) {
        if (src_bf16) pack_a_kernel<3, true><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
        else pack_a_kernel<3, false><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
    } else {
        if (src_bf16) pack_a_kernel<0, true><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
        else pack_a_kernel<0, false><<<grid, 256, 0, s>>>(x, tt, kk, mt, kb, o);
    }
    return hipGetLastError();
}

namespace {

constexpr int WG_NT = GEMM_WG_NT;
constexpr int AR = 4;      // blocks of A fragments held ahead (a whole K-step: two starve the FP8 shapes, whose activations do not stay in L2)

}  // namespace

// grid: (row groups of 128, token groups of 256). apk: packed activations [mtiles][kblocks][64][16 B] with
// kblocks = 4 * steps. OUT_BF16: y is bf16 [t][n_out], else f32.
// With gridDim.z > 1 the K-steps are split over z and each slice writes its partial sums as f32 to
// yv + z * t * n_out (a second kernel adds the slices in order).
// FMT: FMT_Q4M (tile-packed MLX 4-bit), FMT_Q8_0 / FMT_Q8F / FMT_Q4_K / FMT_Q6_K (their tile records) or FMT_FP8 (e4m3 bytes with 128 x 128 block scales: the bytes are
// exact in bf16, the block scale multiplies in f32 before the rounding, and a lane takes 32 consecutive row bytes
// per step, which pack_a's mode 2 mirrors on the activation side).
// (Eight waves of one token tile: two workgroups share a CU if they take at most 128 registers. The 8-bit formats would spill 24 to 40
// bytes, 33.6 -> 43.9 us on 14336 -> 4096: they keep a CU to a workgroup.)
template <int FMT, bool OUT_BF16, int NV, int WAVES, int NT>
__global__ __launch_bounds__(64 * WAVES, WAVES == 4 ? 1 : NV == 1 && !q8_format(FMT) ? 4 : 2) void gemm_bf16_kernel(WeightView w, const uint4* __restrict__ apk, uint32_t t, uint32_t mtiles,
                                                        void* __restrict__ yv) {
    extern __shared__ uint4 bfrag[];  // [2][4 blocks][NT row tiles][64 lanes]
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n = lane & 15;
    constexpr int DT = (NT + WAVES - 1) / WAVES;  // row tiles a wave dequantizes
    const uint32_t all_steps = (w.n_in + 127) / 128, kblocks = 4 * all_steps;  // == t4m_steps(n_in)
    const uint32_t per_z = (all_steps + gridDim.z - 1) / gridDim.z;
    const uint32_t step0 = blockIdx.z * per_z;              // this slice's K-steps: step0 .. step0 + nsteps
    const uint32_t nsteps = min(all_steps, step0 + per_z) - step0;
    const uint32_t ntiles = row_tiles(w.n_out);
    const uint32_t nt0 = blockIdx.x * NT;               // first row tile of the workgroup
    // the wave's token tiles: mt0, mt0 + WAVES, ... (NV of them)
    const uint32_t mt0 = blockIdx.y * (WAVES * NV) + wave;

    // the row tiles this wave dequantizes (with NT = 7 the eighth wave has none)
    const bool has_tile = NT == DT * WAVES || wave < (uint32_t)NT;
    uint32_t tile[DT];
    const uint8_t* wbase[DT];
#pragma unroll
    for (int i = 0; i < DT; i++) {
        tile[i] = min(nt0 + DT * wave + i, ntiles - 1);
        wbase[i] = tile_records<FMT>(w, tile[i], lane);
    }
    // A fragments of the wave's token tiles (tiles past the end repeat the last one; their rows are not stored)
    const uint4* abase[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) abase[i] = apk + ((size_t)min(mt0 + WAVES * i, mtiles - 1) * kblocks + 4 * step0) * 64;  // (the same in every lane)

    f32x4 acc[NV][NT];
#pragma unroll
    for (int i = 0; i < NV; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // `s`: a step of this slice
    auto load_raw = [&](RawTile& r, int i, uint32_t s) {
        if (has_tile) load_tile<FMT>(r, w, wbase[i], tile[i], step0 + s, lane);
    };
    auto dequant = [&](const RawTile& r, int i, uint32_t buf, uint32_t s) {  // the wave's row tile i, 4 blocks
        if (!has_tile) return;
        uint4* dst = bfrag + ((size_t)(buf * 4) * NT + DT * wave + i) * 64 + lane;  // block b: + b * NT * 64
#pragma unroll
        for (int b = 0; b < 4; b++) dst[b * NT * 64] = tile_block<FMT>(r, w, b, step0 + s, lane);
    };
    auto read_b = [&](uint4* dst, uint32_t buf, uint32_t b) {
#pragma unroll
        for (int j = 0; j < NT; j++) dst[j] = bfrag[((buf * 4 + b) * NT + j) * 64 + lane];
    };
    auto read_a = [&](uint4* dst, uint32_t blk) {  // the A fragments of block `blk` of this slice
#pragma unroll
        for (int i = 0; i < NV; i++) {
            // the block's base is the same in every lane: kept in scalar registers, the request takes it with the lane's 32-bit offset
            const uint64_t pa = reinterpret_cast<uint64_t>(abase[i] + (size_t)blk * 64);
            const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)pa), hi = __builtin_amdgcn_readfirstlane((uint32_t)(pa >> 32));
            dst[i] = __builtin_bit_cast(uint4, reinterpret_cast<const __attribute__((address_space(1))) u32x4g*>(((uint64_t)hi << 32) | lo)[lane]);
        }
    };
    // LDS traffic only: outstanding global loads (the prefetches) stay in flight across the barrier
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // B fragments are read from LDS one block ahead of the MFMAs that consume them; A fragments come from global
    // memory a whole K-step (four blocks, ~2000 MFMA cycles) ahead; the packed records of the next step two blocks
    // before they are dequantized into the other LDS buffer. Each fragment has one home, refilled in place right after
    // its last use.
    RawTile raw[DT];
#pragma unroll
    for (int i = 0; i < DT; i++) load_raw(raw[i], i, 0);
    uint4 a_cur[AR][NV], b_cur[NT];
    const uint32_t last = nsteps - 1, last_blk = 4 * nsteps - 1;
#pragma unroll
    for (int b = 0; b < AR; b++) read_a(a_cur[b], min((uint32_t)b, last_blk));
#pragma unroll
    for (int i = 0; i < DT; i++) dequant(raw[i], i, 0, 0);
#pragma unroll
    for (int i = 0; i < DT; i++) load_raw(raw[i], i, min(1u, last));
    lds_barrier();
    read_b(b_cur, 0, 0);
    // One K-step; every step does the same work, so that the loop is one body whose accumulators stay in place: the
    // records of the next step are dequantized into the other LDS buffer during blocks 0 and 1 (with eight waves block 0
    // by the waves 0-3, block 1 by the waves 4-7, which share their SIMDs with them), block 3 refills from
    // that buffer after the barrier, and a tile of the step after next is requested as soon as its registers are free. Past the end
    // the indices repeat the last step: a little work that nobody reads, instead of separate loop tails.
    for (uint32_t s = 0; s < nsteps; s++) {
        const uint32_t buf = s & 1;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b == 3) lds_barrier();  // the other buffer is complete, and nobody still reads this one
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const bf16x8 bb = __builtin_bit_cast(bf16x8, b_cur[j]);
#pragma unroll
                for (int i = 0; i < NV; i++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a_cur[b % AR][i]), bb, acc[i][j], 0, 0, 0);
                if (b < 3) b_cur[j] = bfrag[((buf * 4 + b + 1) * NT + j) * 64 + lane];
                else b_cur[j] = bfrag[(((buf ^ 1) * 4) * NT + j) * 64 + lane];
            }
            read_a(a_cur[b % AR], min(4 * s + b + AR, last_blk));
            if (DT == 2 ? b < 2 : b == (int)(wave >> 2)) {
                const int i = DT == 2 ? b & 1 : 0;
                dequant(raw[i], i, buf ^ 1, min(s + 1, last));
                // (Left to itself the compiler puts the request among the conversions. Q4_K 14336 rows x 2048 tokens 234 us, 226 this way; four
                // waves, medians of 24 calls of up to 64 tokens: Q5_K 0.89 of the time, MXFP4 0.90, Q4_0 0.95, MLX 4-bit, Q8 and Q6_K 0.96
                // to 0.98, Q4_K, FP8 and NVFP4 the same; FP8 past 128 tokens 0.98 to 0.99. The others are no faster.)
                if constexpr (FMT == FMT_Q4_K || WAVES == 4 || (FMT == FMT_FP8 && NV == 2)) __builtin_amdgcn_sched_barrier(0);
                load_raw(raw[i], i, min(s + 2, last));
            }
        }
    }
    // D[token 4 kq + r][row n] per tile
    const uint32_t kq = lane >> 4;
    if (gridDim.z > 1) yv = reinterpret_cast<float*>(yv) + (size_t)blockIdx.z * t * w.n_out;
#pragma unroll
    for (int i = 0; i < NV; i++) {
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const uint32_t row = (nt0 + j) * 16 + n;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t tok = (mt0 + WAVES * i) * 16 + 4 * kq + r;
                if (tok < t && row < w.n_out && mt0 + WAVES * i < mtiles) {
                    if (OUT_BF16) reinterpret_cast<uint16_t*>(yv)[(size_t)tok * w.n_out + row] = f32_to_bf16_bits(acc[i][j][r]);
                    else reinterpret_cast<float*>(yv)[(size_t)tok * w.n_out + row] = acc[i][j][r];
                }
            }
        }
    }
}

// Adds the K slices in order: y = p[0] + p[1] + ... (f32 or bf16 out). VEC outputs per thread (4 when n is a multiple of 4 and
// the buffers are 16-byte aligned). A launch that does not fill the chip is bound by its trips to memory, one per slice where a slice
// is requested when the one before it has been added: BATCH requests eight, four, two and one at a time, the sums as they were
// (16 slices of 17 to 49 tokens, rows of 4096 and of 4095 floats 4.8-5.3 -> 3.9-4.1 us; 8 slices of 65 to 129 tokens, 4096 floats
// 4.8-5.0 -> 4.2-4.4, 4095 floats, one output a thread, 4.8-6.0 -> 4.1-4.5).
template <bool OUT_BF16, int VEC, bool BATCH>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ p, size_t n, uint32_t slices, void* __restrict__ yv) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    if (i >= n) return;
    float v[VEC];
#pragma unroll
    for (int k = 0; k < VEC; k++) v[k] = -0.0f;  // (the zero that leaves every first term as it is)
    uint32_t z = 0;
    auto add = [&](auto many) {
        constexpr int M = decltype(many)::value;
        float b[M][VEC];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float* at = p + (size_t)(z + m) * n + i;
            if constexpr (VEC == 4) {
                const float4 f = *reinterpret_cast<const float4*>(at);
                b[m][0] = f.x; b[m][1] = f.y; b[m][2] = f.z; b[m][3] = f.w;
            } else {
                b[m][0] = *at;
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int k = 0; k < VEC; k++) v[k] += b[m][k];
        z += M;
    };
    if constexpr (BATCH) {
        while (slices - z >= 8) add(std::integral_constant<int, 8>{});
        if ((slices - z) & 4) add(std::integral_constant<int, 4>{});
        if ((slices - z) & 2) add(std::integral_constant<int, 2>{});
        if ((slices - z) & 1) add(std::integral_constant<int, 1>{});
    } else {
        while (z < slices) add(std::integral_constant<int, 1>{});
    }
    if constexpr (VEC == 4) {
        if (OUT_BF16) {
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(yv) + i) =
                make_uint2(f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16), f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16));
        } else {
            *reinterpret_cast<float4*>(reinterpret_cast<float*>(yv) + i) = make_float4(v[0], v[1], v[2], v[3]);
        }
    } else if (OUT_BF16) {
        reinterpret_cast<uint16_t*>(yv)[i] = f32_to_bf16_bits(v[0]);
    } else {
        reinterpret_cast<float*>(yv)[i] = v[0];
    }
}

// Four outputs a thread: past 1.4 million of them the waves in flight cover the trips, and the plain loop streams better (4096 floats x 321
// tokens, 4 slices 5.56 us plain, 5.44 batched; 385 tokens 5.76 and 5.88; 512 tokens of the 14336-column matrix 7.2 and 7.9).
// One output a thread: 4 slices of 449 tokens 7.9 plain, 7.7 batched, and at most 2 % apart beyond.
static void run_gemm_reduce(const float* partial, size_t n, uint32_t slices, void* y, bool out_bf16, hipStream_t s) {
    const bool wide = n % 4 == 0 && reinterpret_cast<uintptr_t>(partial) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
    const unsigned grid = (unsigned)((n / (wide ? 4 : 1) + 255) / 256);
    auto go = [&](auto kern) { kern<<<grid, 256, 0, s>>>(partial, n, slices, y); };
    if (!wide) out_bf16 ? go(gemm_reduce_kernel<true, 1, true>) : go(gemm_reduce_kernel<false, 1, true>);
    else if (n <= 1400000) out_bf16 ? go(gemm_reduce_kernel<true, 4, true>) : go(gemm_reduce_kernel<false, 4, true>);
    else out_bf16 ? go(gemm_reduce_kernel<true, 4, false>) : go(gemm_reduce_kernel<false, 4, false>);
}

static GemmPlan gemm_plan(const WeightView& w, size_t mtiles) { return gemm_plan(w.fmt, w.n_out, w.n_in, mtiles); }

uint32_t gemm_k_slices(const WeightView& w, size_t mtiles) { return gemm_plan(w, mtiles).slices; }

namespace {
template <int FMT, int NV, int WAVES, int NT>
hipError_t run_gemm_bf16_nv(const WeightView& w, const void* apk, size_t t, size_t mtiles, void* y, bool out_bf16, float* partial,
                         hipStream_t s) {
    const uint32_t slices = gemm_k_slices(w, mtiles);
    dim3 grid((row_tiles(w.n_out) + NT - 1) / NT, (unsigned)((mtiles + WAVES * NV - 1) / (WAVES * NV)), slices);
    const size_t lds = 2 * 4 * NT * 64 * 16;  // 64 KiB with 8 row tiles
    const bool direct_bf16 = out_bf16 && slices == 1;
    void* dst = slices > 1 ? static_cast<void*>(partial) : y;
    hipError_t e = hipSuccess;
    auto go = [&](auto kern) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e == hipSuccess) kern<<<grid, 64 * WAVES, lds, s>>>(w, static_cast<const uint4*>(apk), (uint32_t)t, (uint32_t)mtiles, dst);
    };
    span_start(s);
    if (direct_bf16) go(gemm_bf16_kernel<FMT, true, NV, WAVES, NT>);
    else go(gemm_bf16_kernel<FMT, false, NV, WAVES, NT>);
    if (e != hipSuccess) return e;
    e = hipGetLastError();
    span_stop(s);
    if (e != hipSuccess || slices == 1) return e;
    run_gemm_reduce(partial, t * (size_t)w.n_out, slices, y, out_bf16, s);
    return hipGetLastError();
}
template <int FMT>
hipError_t run_gemm_bf16(const WeightView& w, const void* apk, size_t t, size_t mtiles, void* y, bool out_bf16, float* partial,
                         hipStream_t s) {
    if (gemm_waves(mtiles) == 4) return run_gemm_bf16_nv<FMT, 1, 4, WG_NT>(w, apk, t, mtiles, y, out_bf16, partial, s);
    if (gemm_nv(mtiles) == 1) return run_gemm_bf16_nv<FMT, 1, 8, WG_NT>(w, apk, t, mtiles, y, out_bf16, partial, s);
    if (gemm_plan(w, mtiles).nt == 7) return run_gemm_bf16_nv<FMT, 2, 8, 7>(w, apk, t, mtiles, y, out_bf16, partial, s);
    return run_gemm_bf16_nv<FMT, 2, 8, WG_NT>(w, apk, t, mtiles, y, out_bf16, partial, s);
}
}  // namespace

hipError_t launch_gemm_reduce(const float* partial, size_t n, uint32_t slices, void* y, bool out_bf16, hipStream_t s) {
    if (!n) return hipSuccess;
    run_gemm_reduce(partial, n, slices, y, out_bf16, s);
    return hipGetLastError();
}

// `partial`: scratch of slices * t * n_out floats when gemm_k_slices() > 1.
// The formats the kernel dequantizes: tile-packed MLX 4-bit and Q4_0, Q8_0 / Q8, Q4_K, Q6_K, and FP8 rows of whole 128-column
// steps with scale blocks of 16 k rows x 128 k columns.
bool gemm_bf16_ok(const WeightView& w) {
    if (t4_geometry(w.fmt) || q8_format(w.fmt)) return true;
    if (k45_format(w.fmt) || w.fmt == FMT_Q6_K) return w.n_in % 256 == 0;
    return w.fmt == FMT_FP8 && w.br % 16 == 0 && w.bc % 128 == 0 && w.n_in % 128 == 0;
}
// pack_a's MODE for the format's fragments
int gemm_bf16_pack_mode(const WeightView& w) { return t4_geometry(w.fmt) ? 1 : w.fmt == FMT_FP8 ? 2 : w.fmt == FMT_Q6_K ? 3 : 0; }

hipError_t launch_gemm_bf16(const WeightView& w, const void* apk, size_t t, size_t mtiles, void* y, bool out_bf16, float* partial,
                            hipStream_t s) {
    if (!gemm_bf16_ok(w)) return hipErrorInvalidValue;
    switch (w.fmt) {
        case FMT_Q4M: return run_gemm_bf16<FMT_Q4M>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q40: return run_gemm_bf16<FMT_Q40>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_MXFP4: return run_gemm_bf16<FMT_MXFP4>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_NVFP4: return run_gemm_bf16<FMT_NVFP4>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q8_0: return run_gemm_bf16<FMT_Q8_0>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q8F: return run_gemm_bf16<FMT_Q8F>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q4_K: return run_gemm_bf16<FMT_Q4_K>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q5_K: return run_gemm_bf16<FMT_Q5_K>(w, apk, t, mtiles, y, out_bf16, partial, s);
        case FMT_Q6_K: return run_gemm_bf16<FMT_Q6_K>(w, apk, t, mtiles, y, out_bf16, partial, s);
        default: return run_gemm_bf16<FMT_FP8>(w, apk, t, mtiles, y, out_bf16, partial, s);
    }
}

}  // namespace oxhip

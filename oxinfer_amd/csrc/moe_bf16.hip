// Grouped expert matmuls of an MoE prefill pass on the bf16 matrix cores (the experts' forward_batched of the
// reference, src/moe.rs:625-828, over MLX 4-bit weights repacked as Q4 blocks, src/quant.rs:518-606).
//
// With a dozen or more routed tokens per expert the integer path (int8 activations, one scale per token and block of
// 32) spends a conversion and two to three multiply-adds per (row, token, block), and those, not the weights' bytes,
// bound it. Here the routed tokens of a chunk (up to 32 rows of one expert, one or two tiles of 16) go in as bf16 and a weight is the bf16
// value 128 + nibble, two of them made by one mask (nibbles 16 bits apart, | 0x4300). The matrix cores form
//     D = sum (128 + nib) x - 136 sum x = sum (nib - 8) x
// in f32 (the second term is what the accumulator starts from), per group of 64 columns in MLX 4-bit, per block of 32 in the others,
// and y += d D costs one multiply-add per (row, token, group). Codes and single products are exact; the sums are rounded, and what cancels in
// them leaves an error of the order of 2^-24 x 136 sum |x| (Q8_0: 2^-24 x 2304 sum |x|). The offsets of MLX 4-bit and Q4_K, off sum x, are
// one more matrix instruction in f32 (K = four groups or blocks). MXFP4 goes in as 128 + 12 + the doubled E2M1 value. Q8_0's code q as the byte m = q + 128 =
// 16 H + L, both nibbles as 128 + nibble in two matrix instructions: sum q x = 16 D_H + (D_L - 2304 sum x).
// This is the reference's own prefill form: from 8 rows on its
// experts run a grouped f32 GEMM over exact activations with Act::scalar between the two (src/moe.rs:735-827,
// matmul_quant_grouped, src/kernels.rs:195-279); the results here differ from it by the bf16 rounding of the
// activations. The integer path stays the one for decode, where the reference quantizes the activations too.
//
// What bounds it: instruction issue (82 of 203 thousand cycles per SIMD were vector instructions and matrix instructions, half of a wave's time
// waiting, before the steps named below) and the rounds of workgroups. 128 experts of 2048 / 768, 256 tokens, routing to combination, before
// (chunks of 16 rows, an expert with more streamed and unpacked twice; words met through ds_bpermute; a launch that packed the gathered
// rows) -> this: MLX 4-bit 123.5 -> 103 us, Q4_0 145 -> 104, MXFP4 175 -> 127, Q4_K 153 -> 125, Q8_0 206 -> 177 (the last four with the tracer).
#include "act_body.hpp"
#include "internal.hpp"
#include "layout.hpp"
#include "moe_plan.hpp"
#include "moe_rows.hpp"

namespace oxhip {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <bool STD>
__global__ __launch_bounds__(256) void moe_rows_kernel(const float* __restrict__ x, size_t units, uint4* __restrict__ xb, float* __restrict__ sums) {
    moe_row_unit<STD>(x, (size_t)blockIdx.x * 256 + threadIdx.x, units, xb, sums);
}

// The fused gate / up launch's output: act(gate) * up of the workgroup's rows as the down projection's fragments
// [2 chunk + tile][step of 128 columns][block of 32][lane] x 8 bf16, lane 16 kq + n holding gathered row n of the tile, and the blocks' sums
// [2 chunk + tile][step][16 block + n]. The f32 products go through gated_act_scalar and one rounding.
struct MoeGlu {
    uint32_t inter = 0;      // 0: plain products to `out`
    uint32_t kind = 0;
    float param = 0.0f;
    uint32_t std_out = 0;    // the down projection's records hold consecutive columns per lane (Q8_0, Q4_K)
    uint4* frag = nullptr;
    float* sums = nullptr;
};
// Where a chunk's rows come from: rows of x (moe_row_unit) through `rowmap`, or the fragments of a MoeGlu.
struct MoeRows {
    const uint4* x = nullptr;
    const float* sums = nullptr;
    const int* rowmap = nullptr;  // nullptr: fragments
};

// Which (run of row tiles gx, chunk c) a workgroup of the one-dimensional grid takes. Workgroups go to the 8 XCDs in turn
// (linear id mod 8), and each XCD has an L2 of its own; an expert with more than 32 routed rows has several chunks, each
// of which streams the expert's rows again. Items are numbered (gx, c) with c fastest, so that the chunks of one expert
// are neighbours, and XCD k takes the k-th eighth of them in order: workgroups that read the same weights start
// together on the same XCD, and all but the first find them in its L2 instead of asking HBM again. False: no item.
__device__ __forceinline__ bool moe_bf16_item(uint32_t nx, uint32_t nch, uint32_t* gx, uint32_t* c) {
    const uint32_t total = nx * nch, per = (total + 7) >> 3;
    const uint32_t xcd = blockIdx.x & 7, q = blockIdx.x >> 3, v = xcd * per + q;
    if (q >= per || v >= total) return false;
    *gx = __builtin_amdgcn_readfirstlane(v / nch);  // (a division is vector work: without this its result, and all the addresses, would sit in vector registers)
    *c = v - *gx * nch;
    return true;
}

// A request at `voff` bytes past an address that is the same in every lane: the address in scalar registers, 32 bits a lane. (Left to
// itself the compiler makes a 64-bit address per lane of each stream ahead of the loop, and the loop spills.)
template <class T>
__device__ __forceinline__ T gload_at(gbytes base, uint32_t voff) {
    const uint64_t b = (uint64_t)base;
    const uint64_t u = (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
    return gload<T>((gbytes)u + voff);
}

constexpr uint32_t PHASE = MOE_PHASE;
constexpr uint32_t UNIT_LDS = 4096 + 512;  // bytes of one: fragments and sums

// One token tile (TT = 1: up to 16 rows) or two of a chunk; see moe_bf16_kernel.
template <int RT, int FMT, int TT, bool REP>
__device__ __forceinline__ void moe_bf16_body(const WeightView& w, const uint8_t* expert, uint32_t first, uint32_t rows, uint32_t c, uint32_t gx0, const MoeRows& in,
                                              uint32_t kw, uint32_t runs, const MoeGlu& glu, float* __restrict__ out, float* lds) {
    const uint32_t nrep = REP ? runs : 1;
    constexpr bool STD = std_columns(FMT), Q8 = FMT == FMT_Q8_0, PER32 = FMT != FMT_Q4M;  // PER32: a scale per block of 32 instead of a scale and an offset per 64
    constexpr uint32_t P = PHASE / TT;  // steps of a phase
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n = lane & 15, kq = lane >> 4;
    const uint32_t nsteps = w.n_in / 128, ntiles = row_tiles(w.n_out);
    const uint32_t kwsh = (uint32_t)__builtin_ctz(kw), ng = 8u >> kwsh, rg = wave >> kwsh, kwave = wave & (kw - 1);
    // (with the activation fused: the first half of the row groups takes gate tiles, the second the up tiles of the same rows)
    const uint32_t half = ng >> 1, gtiles = glu.inter / 16;
    const uint32_t tend = glu.inter ? gtiles : ntiles, tadd = glu.inter && rg >= half ? gtiles : 0u;
    const gbytes base = as_global(expert);
    gbytes wp[RT];  // (of the run of row tiles that requests go to)
    constexpr uint32_t REC = FMT == FMT_MXFP4 ? T4X_REC : T4M_REC;
    const size_t tile_bytes = Q8 ? (size_t)t8_steps(w.n_in) * T8_REC : FMT == FMT_Q4_K ? (size_t)tk4_sbs(w.n_in) * TK4_REC : (size_t)nsteps * REC;
    auto point_at = [&](uint32_t gx) {
        const uint32_t tile0 = !glu.inter ? (gx * ng + rg) * RT : (gx * half + (rg < half ? rg : rg - half)) * RT;
#pragma unroll
        for (int r = 0; r < RT; r++) wp[r] = base + (size_t)(min(tile0 + r, tend - 1) + tadd) * tile_bytes;
    };
    point_at(gx0 * nrep);
    const uint32_t cnt = (nsteps - kwave + kw - 1) >> kwsh, ilast = cnt - 1;  // kw <= nsteps

    struct St {
        u32x4 w[RT];
        u32x4 w2[Q8 ? RT : 1];     // Q8_0: the step's second record of 64 columns
        uint32_t sc[STD ? RT : 1];  // Q8_0, Q4_K: the row's scale words of the step, one kind per lane group
    };
    // every request is unconditional (past the end the last step again): the compiler then knows how many are in flight
    auto load = [&](St& st, uint32_t i) {
        const uint32_t s = kwave + kw * min(i, ilast);
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if constexpr (Q8) {
                const gbytes rec = wp[r] + (size_t)(2 * s) * T8_REC;
                st.w[r] = gload_at<u32x4>(rec, 16 * lane);
                st.w2[r] = gload_at<u32x4>(rec, T8_REC + 16 * lane);
                st.sc[r] = gload_at<uint32_t>(rec, (kq & 1) * T8_REC + 1024 + 4 * n);
            } else if constexpr (FMT == FMT_Q4_K) {
                const gbytes rec = wp[r] + (size_t)(s >> 1) * TK4_REC;
                st.w[r] = gload_at<u32x4>(rec + (s & 1) * 1024, 16 * lane);
                st.sc[r] = gload_at<uint32_t>(rec, kq == 0 ? 2048 + 16 * n + 4 * (s & 1) : kq == 1 ? 2048 + 16 * n + 8 + 4 * (s & 1) : 2304 + 4 * n);
            } else {
                st.w[r] = gload_at<u32x4>(wp[r] + (size_t)s * REC, 16 * lane);
            }
        }
    };
    // A T4M record's scale words (per row: the two groups' f16 scales at +1024, their bf16 offsets at +1088; Q4_0: four f16 scales; MXFP4: one
    // word of four E8M0 bytes): a request costs the memory pipeline the same for 64 bytes as for 1 KiB, so one request per row tile serves two
    // steps: lane group kq asks for word kq & 1 of step i + (kq >> 1), and at each step every lane takes its row's words from those lanes.
    uint32_t scl[STD ? 1 : RT];
    auto load_scales = [&](uint32_t i) {
        if constexpr (!STD) {
            const uint32_t i0 = min(i, ilast), s = kwave + kw * i0, at = kw * (min(i0 + (kq >> 1), ilast) - i0) * REC + 1024 + (FMT == FMT_MXFP4 ? 0 : 64 * (kq & 1)) + 4 * n;
#pragma unroll
            for (int r = 0; r < RT; r++) scl[r] = gload_at<uint32_t>(wp[r] + (size_t)s * REC, at);
        }
    };
    // The rows' words meet all lane groups by swaps of 16 and 32 lanes: two instructions of the vector unit for two words, where a
    // lane-to-lane read through the LDS pipe costs a trip of its own in front of every step (128 MLX 4-bit experts, 256 tokens: the gate / up
    // launch 81 us with ds_bpermute, 64 without).
    auto swap16 = [](uint32_t x, uint32_t& even, uint32_t& odd) {  // rows of 16 lanes {0, 0, 2, 2} and {1, 1, 3, 3} of x
        const auto v = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        even = v[0], odd = v[1];
    };
    auto swap32 = [](uint32_t x, uint32_t& lo, uint32_t& hi) {  // the lower and the upper half of x, twice each
        const auto v = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        lo = v[0], hi = v[1];
    };
    auto half_of = [](uint32_t v, uint32_t h) { return f16_bits_to_f32((uint16_t)(h ? v >> 16 : v & 0xFFFF)); };
    // the scale of block `b` of the step (opaque, so that the products take it as f32: with the f16 inside the multiply-add that is
    // an instruction of 1.6 times the time)
    auto scale = [&](const uint32_t* W, int b) -> float {
        float d;
        if constexpr (FMT == FMT_Q4M) d = half_of(W[0], b >> 1);
        else if constexpr (FMT == FMT_MXFP4) d = e8m0_half((W[0] >> (8 * b)) & 0xFF);
        else if constexpr (FMT == FMT_Q4_K) d = f16_bits_to_f32((uint16_t)(W[2] & 0xFFFF)) * (float)((W[0] >> (8 * b)) & 0xFF);
        else d = half_of(b >> 1 ? W[1] : W[0], b & 1);
        asm("" : "+v"(d));
        return d;
    };
    // The codes go in as the bf16 values 128 + code; BIAS x the activations' sum takes what that adds (and the formats' own zero) out again:
    // it is what the block's products start from, so a sum of sum (code - zero) x costs nothing further.
    constexpr float BIAS = FMT == FMT_Q4_K ? -128.0f : Q8 ? -2304.0f : FMT == FMT_MXFP4 ? -140.0f : -136.0f;
    constexpr bool OFF = FMT == FMT_Q4M || FMT == FMT_Q4_K;  // an offset times the sum besides
    // eight codes, one per nibble (c0: four, c1: four, at bits 0 and 16, shifted by 8 bits 8 and 24), as 128 + code in pack_columns' order
    const uint32_t mlo = 0x000F000Fu;
    uint32_t magic = 0x43004300u;
    asm("" : "+v"(magic));
    auto pair = [&](uint32_t x) { return (uint32_t)__builtin_amdgcn_bitop3_b32(x, mlo, magic, 0xEA); };  // (x & mask) | magic
    auto operand = [&](uint32_t c0, uint32_t c1) {
        const u32x4 wb = {pair(c0), pair(c0 >> 8), pair(c1), pair(c1 >> 8)};
        return __builtin_bit_cast(bf16x8, wb);
    };
    constexpr uint32_t NIB = 0x0F0F0F0Fu;

    // Staging of phase `ph`: 256 pieces of 16 bytes per step and tile. From rows of x: lane bits 0-2 are (kq, block & 1), bits 3-6 the
    // row, bit 7 the block's upper bit, so that a request covers whole lines of eight rows and a thread keeps to one row.
    u32x4* lf = reinterpret_cast<u32x4*>(lds);                       // [step][tile][4][64]
    constexpr uint32_t NB = PER32 ? 4 : 2, NS = 16 * NB;              // sums of a step and tile: [block or group][16 tokens]
    float* ls = lds + PHASE * 1024;                                   // [step][tile][NS], for the offsets
    float* lb = ls + PHASE * 64;                                      // the same times BIAS
    const uint32_t tid = threadIdx.x;
    constexpr int SG = 4, PF = 2;
    St ring[PF];
    uint32_t frow = 0, srow = 0;
    bool flive = true, slive = true;
    if (in.rowmap) {
        const uint32_t fr = ((tid >> 3) & 15) + (TT == 2 ? 16 * ((tid >> 8) & 1) : 0), sr = (tid & 15) + (TT == 2 ? 16 * ((tid / NS) & 1) : 0);
        flive = fr < rows, slive = sr < rows;
        frow = (uint32_t)in.rowmap[first + (flive ? fr : 0)], srow = (uint32_t)in.rowmap[first + (slive ? sr : 0)];
    }
    auto stage = [&](uint32_t ph, bool begin) {
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));  // (or every piece's address would be made ahead of the phases and kept)
        const uint32_t s0 = ph * P, ns = min(P, nsteps - s0), total = ns * TT * 256, stotal = ns * TT * NS;
        float sm[2];
        auto piece = [&](uint32_t u) -> u32x4 {
            const uint32_t st = u >> 8, step = s0 + st / TT, tile = st % TT;
            if (in.rowmap) return reinterpret_cast<const u32x4*>(in.x)[(size_t)frow * (w.n_in / 8) + step * 16 + ((u >> 7) & 1) * 8 + (u & 7)];
            return gload_at<u32x4>(as_global(reinterpret_cast<const uint8_t*>(in.x)) + ((size_t)2 * c * nsteps + s0) * 4096, (tile * nsteps + (step - s0)) * 4096 + 16 * (u & 255));
        };
        for (uint32_t i0 = 0; i0 < total; i0 += 512 * SG) {
            u32x4 t[SG];
#pragma unroll
            for (int k = 0; k < SG; k++) t[k] = piece(min(i0 + 512 * k + tid, total - 1));
            if (i0 == 0) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const uint32_t u = min(512 * k + tid, stotal - 1), st = u / NS, step = s0 + st / TT, tile = st % TT, b = (u % NS) >> 4;
                    const float* at = in.rowmap ? in.sums + (size_t)srow * (w.n_in / 32) + 4 * step + (PER32 ? b : 2 * b)
                                                : in.sums + ((size_t)(2 * c + tile) * nsteps + step) * 64 + (PER32 ? 16 : 32) * b + (u & 15);
                    sm[k] = PER32 ? at[0] : at[0] + at[in.rowmap ? 1 : 16];
                }
                if (begin) {
                    load_scales(0);
#pragma unroll
                    for (int p = 0; p < PF; p++) load(ring[p], (uint32_t)p);
                }
            }
#pragma unroll
            for (int k = 0; k < SG; k++) {
                const uint32_t u = i0 + 512 * k + tid;
                if (u >= total) break;
                if (in.rowmap) lf[(u >> 8) * 256 + 128 * ((u >> 7) & 1) + 64 * ((u >> 2) & 1) + 16 * (u & 3) + ((u >> 3) & 15)] = flive ? t[k] : u32x4{0, 0, 0, 0};
                else lf[u] = t[k];
            }
        }
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (512 * k + tid < stotal) {
                const float v = slive ? sm[k] : 0.0f;
                if (OFF) ls[512 * k + tid] = v;
                lb[512 * k + tid] = BIAS * v;
            }
    };

    f32x4 acc[RT][TT];
    // The offsets' terms: one f32 matrix instruction (rows = tokens, K = 4) for the four blocks of a step (Q4_K) or the groups of two steps
    // (MLX 4-bit; `second`: there is a second one).
    auto offsets = [&](int r, float cc, uint32_t sl, bool second) {
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            float e;
            if constexpr (PER32) e = ls[(sl * TT + tt) * NS + lane];
            else {
                const float v = ls[((sl + (second ? kw * (kq >> 1) : 0)) * TT + tt) * NS + (lane & 31)];
                e = second || kq < 2 ? v : 0.0f;
            }
            acc[r][tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(e, cc, acc[r][tt], 0, 0, 0);
        }
    };
    // T4M records: what two steps' words come to, the first step's in [0]
    uint32_t pw[STD ? 1 : RT][2][FMT == FMT_Q40 ? 2 : 1];
    auto unfold = [&](uint32_t sl, bool second) {
        if constexpr (!STD) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                uint32_t w0, w1;
                swap16(scl[r], w0, w1);  // (either step's first words in its half of the lanes, and its second)
                swap32(w0, pw[r][0][0], pw[r][1][0]);
                if constexpr (FMT == FMT_Q40) swap32(w1, pw[r][0][1], pw[r][1][1]);
                if constexpr (FMT == FMT_Q4M) offsets(r, __uint_as_float(kq & 1 ? w1 & 0xFFFF0000u : w1 << 16), sl, second);
            }
        }
    };
    // `sl`: the step's place in its phase
    auto compute = [&](const St& st, int odd, uint32_t sl) {
        uint32_t W[RT][3];
        if constexpr (STD) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                uint32_t lo, hi, rest;
                swap32(st.sc[r], lo, hi);
                swap16(lo, W[r][0], W[r][1]);
                if constexpr (FMT == FMT_Q4_K) {
                    swap16(hi, W[r][2], rest);
                    offsets(r, -(f16_bits_to_f32((uint16_t)(W[r][2] >> 16)) * (float)((W[r][1] >> (8 * kq)) & 0xFF)), sl, false);
                }
            }
        }
#pragma unroll
        for (int g = 0; g < 2; g++) {
            bf16x8 a[TT][2];
            f32x4 bias[TT][PER32 ? 2 : 1];
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
#pragma unroll
                for (int e = 0; e < 2; e++) a[tt][e] = __builtin_bit_cast(bf16x8, lf[((sl * TT + tt) * 4 + 2 * g + e) * 64 + lane]);
#pragma unroll
                for (int e = 0; e < (PER32 ? 2 : 1); e++) bias[tt][e] = *reinterpret_cast<const f32x4*>(lb + (sl * TT + tt) * NS + (PER32 ? 32 * g + 16 * e : 16 * g) + 4 * kq);
            }
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const uint32_t* wr = STD ? W[r] : pw[STD ? 0 : r][odd];
                f32x4 D[TT];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int b = 2 * g + e;
                    if constexpr (Q8) {
                        const u32x4 v = g ? st.w2[r] : st.w[r];
                        const uint32_t c0 = v[2 * e] ^ 0x80808080u, c1 = v[2 * e + 1] ^ 0x80808080u;
                        const bf16x8 hi = operand(c0 >> 4, c1 >> 4), lo = operand(c0, c1);
                        const float d = scale(wr, b);
#pragma unroll
                        for (int tt = 0; tt < TT; tt++) {
                            const f32x4 DH = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tt][e], hi, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                            const f32x4 DL = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tt][e], lo, bias[tt][e], 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 4; i++) acc[r][tt][i] = fmaf(d, fmaf(16.0f, DH[i], DL[i]), acc[r][tt][i]);
                        }
                    } else {
                        bf16x8 wb;
                        if constexpr (FMT == FMT_Q4_K) {  // block b = 2 g + e: the low (e = 0) or high nibbles of the byte pair g
                            wb = operand(st.w[r][2 * g] >> (4 * e), st.w[r][2 * g + 1] >> (4 * e));
                        } else if constexpr (FMT == FMT_MXFP4) {  // table codes -> their doubled values + 12 (0 .. 24)
                            const uint32_t lo = mxfp4_values<12>(st.w[r][b] & NIB), hi = mxfp4_values<12>((st.w[r][b] >> 4) & NIB);
                            const u32x4 v = {__builtin_amdgcn_perm(magic, lo, 0x05020500u), __builtin_amdgcn_perm(magic, lo, 0x05030501u),
                                             __builtin_amdgcn_perm(magic, hi, 0x05020500u), __builtin_amdgcn_perm(magic, hi, 0x05030501u)};
                            wb = __builtin_bit_cast(bf16x8, v);
                        } else {  // byte j of dword b: low nibble = position 4 kq + j, high nibble = position 16 + 4 kq + j
                            wb = operand(st.w[r][b], st.w[r][b] >> 4);
                        }
#pragma unroll
                        for (int tt = 0; tt < TT; tt++) D[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tt][e], wb, PER32 || e == 0 ? bias[tt][PER32 ? e : 0] : D[tt], 0, 0, 0);
                        if (PER32 || e == 1) {
                            const float d = scale(wr, b);
#pragma unroll
                            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                                for (int i = 0; i < 4; i++) acc[r][tt][i] = fmaf(d, D[tt][i], acc[r][tt][i]);
                        }
                    }
                }
            }
        }
    };
    const uint32_t nph = (nsteps + P - 1) / P, even = (cnt + 1) & ~1u;
    for (uint32_t rep = 0; rep < nrep; rep++) {
        const uint32_t gx = gx0 * nrep + rep;
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) acc[r][tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t i = 0;
        for (uint32_t ph = 0; ph < nph; ph++) {
            if (rep == 0 || nph > 1) {  // (rows staged whole serve all runs)
                if (rep + ph) __syncthreads();
                stage(ph, rep + ph == 0);
                __syncthreads();
            }
            // (kw divides a phase's steps, and leaves each wave an even number of them)
            const uint32_t iend = min(even, (ph + 1) * (P >> kwsh));
            for (; i < iend; i += PF) {
                if (i < cnt) unfold(kwave + kw * i - ph * P, i + 1 < cnt);
                // (the run's last two steps make room for the next run's first)
                const bool over = i + PF >= even && rep + 1 < nrep;
                const uint32_t next = over ? 0 : i + PF;
                if (over) point_at(gx + 1);
#pragma unroll
                for (int p = 0; p < PF; p++) {
                    if (i + p < cnt) compute(ring[p], p, kwave + kw * (i + p) - ph * P);
                    load(ring[p], next + p);
                }
                load_scales(next);
            }
        }
        if (kw > 1 || glu.inter) break;  // (one run: the waves' sums meet in LDS)
        // D[token 4 kq + e][row n]
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const uint32_t row = ((gx * ng + rg) * RT + r) * 16 + n;
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t tok = 16 * tt + 4 * kq + e;
                    if (tok < rows && row < w.n_out) out[(size_t)(first + tok) * w.n_out + row] = acc[r][tt][e];
                }
        }
    }
    if (kw == 1 && !glu.inter) return;
    const uint32_t gx = gx0;
    __syncthreads();  // the sums overwrite the fragments
    f32x4* red = reinterpret_cast<f32x4*>(lds);  // [wave][RT][TT][64]
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) red[((wave * RT + r) * TT + tt) * 64 + lane] = acc[r][tt];
    __syncthreads();
    if (glu.inter) {  // uniform over the launch
        const float* rf = reinterpret_cast<const float*>(red);
        const uint32_t blocks = half * RT / 2, osteps = glu.inter / 128;  // blocks of 32 rows of the workgroup
        for (uint32_t idx = tid; idx < blocks * TT * 64; idx += 512) {
            const uint32_t l = idx & 63, tile = (idx >> 6) % TT, bl = (idx >> 6) / TT, m = l & 15, q = l >> 4;
            const uint32_t blk = gx * blocks + bl;
            if (blk >= glu.inter / 32) break;  // (uniform over a wave)
            uint4 pk = make_uint4(0, 0, 0, 0);
            float sum = 0.0f;
            if (m + 16 * tile < rows) {
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t col = 32 * bl + (glu.std_out ? 8 * q + j : 4 * q + (j & 3) + 16 * (j >> 2));
                    const uint32_t t = col >> 4, g = t / RT, r = t % RT;
                    float gate = 0.0f, up = 0.0f;
                    for (uint32_t k = 0; k < kw; k++) {
                        const uint32_t at = ((((g * kw + k) * RT + r) * TT + tile) * 64 + 16 * (m >> 2) + (col & 15)) * 4 + (m & 3);
                        const float a = rf[at], b = rf[at + half * kw * RT * TT * 256];
                        gate = k ? gate + a : a;
                        up = k ? up + b : b;
                    }
                    v[j] = gated_act_scalar(gate, up, glu.kind, glu.param);
                }
                pk = pack_columns(v, &sum);
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            const size_t at = (size_t)(2 * c + tile) * osteps + (blk >> 2);
            glu.frag[at * 256 + (blk & 3) * 64 + l] = pk;
            if (q == 0) glu.sums[at * 64 + (blk & 3) * 16 + m] = sum;
        }
        return;
    }
    // D[token 4 kq + i][row n]: thread (group, r, tile, lane) adds the group's waves in order and stores its four tokens
    for (uint32_t idx = tid; idx < ng * RT * TT * 64; idx += 512) {
        const uint32_t l = idx & 63, tt = (idx >> 6) % TT, r = (idx >> 6) / TT % RT, g = (idx >> 6) / (TT * RT);
        const uint32_t tile = (gx * ng + g) * RT + r, row = tile * 16 + (l & 15);
        if (tile >= ntiles || row >= w.n_out) continue;
        f32x4 sum = red[((g * kw * RT + r) * TT + tt) * 64 + l];
        for (uint32_t k = 1; k < kw; k++) {
            const f32x4 v = red[(((g * kw + k) * RT + r) * TT + tt) * 64 + l];
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] += v[e];
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t tok = 16 * tt + 4 * (l >> 4) + e;
            if (tok < rows) out[(size_t)(first + tok) * w.n_out + row] = sum[e];
        }
    }
}

// Workgroup: 8 waves = 8 / kw groups of RT row tiles x kw waves that split the K steps (wave v takes steps v, v + kw, ...)
// and meet in LDS in wave order. A workgroup's item (moe_bf16_item): a run of (8 / kw) RT row tiles of a chunk {expert, first row, rows <= 32}.
// The chunk's rows (4 KiB per step and tile of 16) are staged into LDS, 64 KiB at a time: all eight waves multiply the same rows (each wave
// asking memory for them costs more than the weights), and two workgroups share a CU. out [gathered row][n_out] f32.
// REP: an item is `nrep` such runs of row tiles, one after the other over the same staged rows (kw = 1, no activation). (These forms keep 37
// to 76 scalar registers in vector lanes, the others 0 to 23: the bodies of one and two token tiles, the activation and the waves' join are
// one kernel. No form spills vector registers.)
template <int RT, int FMT, bool REP>
__global__ __launch_bounds__(512, 4) void moe_bf16_kernel(WeightView w, const uint8_t* const* __restrict__ bases, const int4* __restrict__ chunks,
                                                          const int* __restrict__ nchunks, MoeRows in, uint32_t kw, uint32_t nrep, uint32_t nx, MoeGlu glu,
                                                          float* __restrict__ out) {
    extern __shared__ __align__(16) float lds[];
    uint32_t gx, c;
    if (!moe_bf16_item(nx, (uint32_t)*nchunks, &gx, &c)) return;  // uniform over the workgroup
    // (the same in every lane: kept in scalar registers, as what follows from them then is)
    int4 ch = chunks[c];
    ch.x = __builtin_amdgcn_readfirstlane(ch.x), ch.y = __builtin_amdgcn_readfirstlane(ch.y), ch.z = __builtin_amdgcn_readfirstlane(ch.z);
    const uint64_t eb = reinterpret_cast<uint64_t>(bases[ch.x]);
    const uint8_t* expert = reinterpret_cast<const uint8_t*>((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(eb >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)eb));
    if (ch.z <= 16) moe_bf16_body<RT, FMT, 1, REP>(w, expert, (uint32_t)ch.y, (uint32_t)ch.z, c, gx, in, kw, nrep, glu, out, lds);
    else moe_bf16_body<RT, FMT, 2, REP>(w, expert, (uint32_t)ch.y, (uint32_t)ch.z, c, gx, in, kw, nrep, glu, out, lds);
}

}  // namespace

// (Rows of up to 4096 columns: the form once staged a chunk's rows whole. It stages them in phases now, but longer rows have not been measured
// here against the integer kernels, which they keep.)
bool moe_bf16_ok(const WeightView& w) {
    if (w.n_in % 128 || w.n_in < 128 || w.n_in > 4096) return false;
    return t4m_format(w.fmt) || w.fmt == FMT_Q8_0 || (w.fmt == FMT_Q4_K && w.n_in % 256 == 0);
}
size_t moe_bf16_row_bytes(size_t t, size_t n_in) { return t * n_in * 2 + t * (n_in / 32) * 4; }
size_t moe_bf16_frag_bytes(size_t max_chunks, size_t n_in) { return 2 * max_chunks * (n_in / 128) * (4096 + 256); }

// x [t][n_in] for the gate / up launch over experts like `w`: rows, then their blocks' sums (moe_bf16_row_bytes).
hipError_t launch_moe_rows(const float* x, size_t t, const WeightView& w, void* rows, hipStream_t s) {
    const size_t units = t * w.n_in / 8;
    if (!units) return hipSuccess;
    uint4* xb = static_cast<uint4*>(rows);
    float* sums = reinterpret_cast<float*>(xb + units);
    const unsigned grid = (unsigned)((units + 255) / 256);
    if (std_columns(w.fmt)) moe_rows_kernel<true><<<grid, 256, 0, s>>>(x, units, xb, sums);
    else moe_rows_kernel<false><<<grid, 256, 0, s>>>(x, units, xb, sums);
    return hipGetLastError();
}

namespace {
template <int FMT>
hipError_t run_moe_bf16(const WeightView& w, const GroupView& g, uint32_t max_chunks, const MoeRows& in, const MoeGlu& glu, uint32_t chunks, float* out, hipStream_t s) {
    const MoePlan p = moe_plan(FMT, w.n_out, w.n_in, glu.inter, max_chunks, chunks);
    const size_t lds = PHASE * UNIT_LDS;
    const dim3 grid((p.nx * max_chunks + 7) / 8 * 8);  // every XCD's share of the items (moe_bf16_item), whatever the chunk count turns out to be
    auto go = [&](auto kern) -> hipError_t {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        kern<<<grid, 512, lds, s>>>(w, g.bases, g.chunks, g.nchunks, in, p.kw, p.nrep, p.nx, glu, out);
        return hipGetLastError();
    };
    if constexpr (FMT != FMT_Q8_0) {
        if (p.nrep > 1) return go(moe_bf16_kernel<2, FMT, true>);
        if (p.rt == 3) return go(moe_bf16_kernel<3, FMT, false>);
    }
    return go(moe_bf16_kernel<2, FMT, false>);
}
hipError_t launch_moe_bf16(const WeightView& w, const GroupView& g, uint32_t max_chunks, const MoeRows& in, const MoeGlu& glu, uint32_t chunks, float* out, hipStream_t s) {
    if (!moe_bf16_ok(w) || (glu.inter && (w.n_out != 2 * glu.inter || glu.inter % 128))) return hipErrorInvalidValue;
    if (!max_chunks) return hipSuccess;
    switch (w.fmt) {
        case FMT_Q8_0: return run_moe_bf16<FMT_Q8_0>(w, g, max_chunks, in, glu, chunks, out, s);
        case FMT_Q4_K: return run_moe_bf16<FMT_Q4_K>(w, g, max_chunks, in, glu, chunks, out, s);
        case FMT_Q40: return run_moe_bf16<FMT_Q40>(w, g, max_chunks, in, glu, chunks, out, s);
        case FMT_MXFP4: return run_moe_bf16<FMT_MXFP4>(w, g, max_chunks, in, glu, chunks, out, s);
        default: return run_moe_bf16<FMT_Q4M>(w, g, max_chunks, in, glu, chunks, out, s);
    }
}
}  // namespace

// The gate / up launch over fused experts `w` ([2 inter, h]): `rows` as launch_moe_rows made them, through g.rowmap; the activation is the
// launch's output stage, which writes the fragments (moe_bf16_frag_bytes) for the down projection `down`. `chunks`: as many as are to be
// expected of the max_chunks there may be.
hipError_t launch_moe_bf16_gate(const WeightView& w, const WeightView& down, const GroupView& g, uint32_t max_chunks, uint32_t chunks, const void* rows, size_t t,
                                uint32_t act_kind, float act_param, void* frag, hipStream_t s) {
    const uint4* xb = static_cast<const uint4*>(rows);
    const MoeRows in{xb, reinterpret_cast<const float*>(xb + t * w.n_in / 8), g.rowmap};
    uint4* f = static_cast<uint4*>(frag);
    const MoeGlu glu{down.n_in, act_kind, act_param, std_columns(down.fmt) ? 1u : 0u, f, reinterpret_cast<float*>(f + 2 * (size_t)max_chunks * (down.n_in / 128) * 256)};
    return launch_moe_bf16(w, g, max_chunks, in, glu, chunks, nullptr, s);
}
// The down launch over those fragments: `out` receives the gathered rows' products.
hipError_t launch_moe_bf16_down(const WeightView& w, const GroupView& g, uint32_t max_chunks, uint32_t chunks, const void* frag, float* out, hipStream_t s) {
    const uint4* f = static_cast<const uint4*>(frag);
    const MoeRows in{f, reinterpret_cast<const float*>(f + 2 * (size_t)max_chunks * (w.n_in / 128) * 256), nullptr};
    return launch_moe_bf16(w, g, max_chunks, in, MoeGlu{}, chunks, out, s);
}

}  // namespace oxhip

// The packed weight records of every format as bf16 matrix-core operands: what the prefill GEMMs (gemm.hip, gemm_short.hip) share.
#pragma once
#include "internal.hpp"
#include "layout.hpp"

namespace oxhip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4g __attribute__((ext_vector_type(4)));

namespace {

// the formats in the T4M code geometry (NVFP4's records too: float-stored, so not one of the int8 decode formats)
__host__ __device__ constexpr bool t4_geometry(int f) { return t4m_format(f) || f == FMT_NVFP4; }

// Two f32 -> packed bf16 (round to nearest even) with the hardware conversion, one instruction, no branches.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// Eight unsigned byte codes (the bytes of lo, then of hi) -> 8 bf16 of code * d + c.
template <int K>
__device__ __forceinline__ float byte_f32(uint32_t x) {  // byte K of x as f32: one conversion that selects the byte itself
    float f;
    if constexpr (K == 0) asm("v_cvt_f32_ubyte0_e32 %0, %1" : "=v"(f) : "v"(x));
    else if constexpr (K == 1) asm("v_cvt_f32_ubyte1_e32 %0, %1" : "=v"(f) : "v"(x));
    else if constexpr (K == 2) asm("v_cvt_f32_ubyte2_e32 %0, %1" : "=v"(f) : "v"(x));
    else asm("v_cvt_f32_ubyte3_e32 %0, %1" : "=v"(f) : "v"(x));
    return f;
}
__device__ __forceinline__ uint4 dequant_u8x8(uint32_t lo, uint32_t hi, float d, float c) {
    float f[8];
    f[0] = __builtin_fmaf(byte_f32<0>(lo), d, c);
    f[1] = __builtin_fmaf(byte_f32<1>(lo), d, c);
    f[2] = __builtin_fmaf(byte_f32<2>(lo), d, c);
    f[3] = __builtin_fmaf(byte_f32<3>(lo), d, c);
    f[4] = __builtin_fmaf(byte_f32<0>(hi), d, c);
    f[5] = __builtin_fmaf(byte_f32<1>(hi), d, c);
    f[6] = __builtin_fmaf(byte_f32<2>(hi), d, c);
    f[7] = __builtin_fmaf(byte_f32<3>(hi), d, c);
    return make_uint4(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
}
// One dword of a T4M chunk (4 bytes of one block: low nibbles = elements 4 kq + i, high = 16 + 4 kq + i) -> the
// lane's 8 bf16 of that block.
__device__ __forceinline__ uint4 dequant_q4m(uint32_t w, float d, float c) {
    return dequant_u8x8(w & 0x0F0F0F0Fu, (w >> 4) & 0x0F0F0F0Fu, d, c);
}

// One row tile's records of a step of 128 columns, as a wave holds them between the request and the use.
struct RawTile {
    uint4 c, c2;    // Q4M, Q4_K: one chunk; Q8: the chunks of the step's two records; Q6_K: low nibbles, high bit pairs; FP8: 32 row bytes
    uint32_t m[4];  // the row's scale words (Q4M: scales, offsets; FP8: the block scale's bits)
};
// Where a row tile's records begin (FP8: the lane's bytes of the matrix's first step).
template <int FMT>
__device__ __forceinline__ const uint8_t* tile_records(const WeightView& w, uint32_t tile, uint32_t lane) {
    if constexpr (t4_geometry(FMT)) return w.p0 + (size_t)tile * t4m_steps(w.n_in) * (FMT == FMT_MXFP4 ? T4X_REC : T4M_REC);  // (T4N_REC == T4M_REC)
    else if constexpr (q8_format(FMT)) return w.p0 + (size_t)tile * t8_steps(w.n_in) * (FMT == FMT_Q8F ? T8F_REC : T8_REC);
    else if constexpr (k45_format(FMT)) return w.p0 + (size_t)tile * tk4_sbs(w.n_in) * (FMT == FMT_Q5_K ? TK5_REC : TK4_REC);
    else if constexpr (FMT == FMT_Q6_K) return w.p0 + (size_t)tile * t6k_steps(w.n_in) * T6K_REC;
    else return w.p0 + fp8_offset(w, min(tile * 16 + (lane & 15), w.n_out - 1), 32 * (lane >> 4));
}
// Requests the records of `tile` (which begin at `base`) for the matrix's step `s`. Nothing here may depend on a loaded value, or the
// request would be waited for where it is made.
template <int FMT>
__device__ __forceinline__ void load_tile(RawTile& r, const WeightView& w, const uint8_t* base, uint32_t tile, uint32_t s, uint32_t lane) {
    const uint32_t n = lane & 15;
    if constexpr (FMT == FMT_NVFP4) {  // the row's eight sub-block scale bytes, and the matrix's scale of this step's columns
        const uint8_t* rec = base + (size_t)s * T4N_REC;
        r.c = *reinterpret_cast<const uint4*>(rec + 16 * lane);
        const uint2 sv = *reinterpret_cast<const uint2*>(rec + 1024 + 8 * n);
        r.m[0] = sv.x;
        r.m[1] = sv.y;
        r.m[2] = w.br ? __float_as_uint(reinterpret_cast<const float*>(w.p1)[(size_t)(min(tile * 16 + n, w.n_out - 1) / w.br) * ((w.n_in + w.bc - 1) / w.bc) + (128 * s) / w.bc])
                      : 0x3F800000u;
    } else if constexpr (t4m_format(FMT)) {
        const uint8_t* rec = base + (size_t)s * (FMT == FMT_MXFP4 ? T4X_REC : T4M_REC);
        r.c = *reinterpret_cast<const uint4*>(rec + 16 * lane);
        r.m[0] = *reinterpret_cast<const uint32_t*>(rec + 1024 + 4 * n);
        if (FMT != FMT_MXFP4) r.m[1] = *reinterpret_cast<const uint32_t*>(rec + 1088 + 4 * n);
    } else if constexpr (q8_format(FMT)) {  // a step of 128 columns is two records of 64 (past the row's last record: that one again, which
                                            // tile_block zeroes)
        constexpr uint32_t REC = FMT == FMT_Q8F ? T8F_REC : T8_REC;
        const uint32_t nrec = t8_steps(w.n_in);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint8_t* rec = base + (size_t)min(2 * s + h, nrec - 1) * REC;
            const uint4 v = *reinterpret_cast<const uint4*>(rec + 16 * lane);
            if (h) r.c2 = v;
            else r.c = v;
            if (FMT == FMT_Q8F) {
                const uint2 sc = *reinterpret_cast<const uint2*>(rec + 1024 + 8 * n);
                r.m[2 * h] = sc.x;
                r.m[2 * h + 1] = sc.y;
            } else {
                r.m[h] = *reinterpret_cast<const uint32_t*>(rec + 1024 + 4 * n);
            }
        }
    } else if constexpr (k45_format(FMT)) {  // half a super-block record: sub-blocks 4 (s & 1) .. + 3
        const uint8_t* rec = base + (size_t)(s >> 1) * (FMT == FMT_Q5_K ? TK5_REC : TK4_REC);
        r.c = *reinterpret_cast<const uint4*>(rec + (s & 1) * 1024 + 16 * lane);
        if (FMT == FMT_Q5_K) r.c2.x = *reinterpret_cast<const uint32_t*>(rec + TK4_REC + (s & 1) * 256 + 4 * lane);
        r.m[0] = *reinterpret_cast<const uint32_t*>(rec + 2048 + 16 * n + 4 * (s & 1));
        r.m[1] = *reinterpret_cast<const uint32_t*>(rec + 2048 + 16 * n + 8 + 4 * (s & 1));
        r.m[2] = *reinterpret_cast<const uint32_t*>(rec + 2304 + 4 * n);
    } else if constexpr (FMT == FMT_Q6_K) {
        const uint8_t* rec = base + (size_t)s * T6K_REC;
        r.c = *reinterpret_cast<const uint4*>(rec + 16 * lane);
        const uint2 hb = *reinterpret_cast<const uint2*>(rec + 1024 + 8 * lane);
        r.c2.x = hb.x;
        r.c2.y = hb.y;
        const uint2 sc = *reinterpret_cast<const uint2*>(rec + 1536 + 8 * n);
        r.m[0] = sc.x;
        r.m[1] = sc.y;
        r.m[2] = *reinterpret_cast<const uint16_t*>(rec + 1664 + 2 * n);
    } else {
        const uint8_t* p = base + (w.group == 1 ? 2048 : 128) * (size_t)s;
        r.c = *reinterpret_cast<const uint4*>(p);
        r.c2 = *reinterpret_cast<const uint4*>(p + fp8_second_chunk(w));
        r.m[0] = __float_as_uint(reinterpret_cast<const float*>(w.p1)[(size_t)(tile * 16 / w.br) * ((w.n_in + w.bc - 1) / w.bc) + (128 * s) / w.bc]);
    }
}
// Block `b` (0..3) of the step as the lane's eight bf16 of the matrix cores' operand; `s`: the step the records belong to.
template <int FMT>
__device__ __forceinline__ uint4 tile_block(const RawTile& r, const WeightView& w, int b, uint32_t s, uint32_t lane) {
    const uint32_t cw[8] = {r.c.x, r.c.y, r.c.z, r.c.w, r.c2.x, r.c2.y, r.c2.z, r.c2.w};
    if constexpr (FMT == FMT_NVFP4) {  // as MXFP4 below with a scale per 16: the low nibbles' sub-block 2 b, the high nibbles' 2 b + 1
        const float g = __uint_as_float(r.m[2]);
        const uint32_t sw = r.m[b >> 1] >> (16 * (b & 1));
        const float d0 = ue4m3_half(sw) * g, d1 = ue4m3_half(sw >> 8) * g;
        const uint32_t lo = mxfp4_values<12>(cw[b] & 0x0F0F0F0Fu), hi = mxfp4_values<12>((cw[b] >> 4) & 0x0F0F0F0Fu);
        const float c0 = -12.0f * d0, c1 = -12.0f * d1;
        return make_uint4(pack_bf16(__builtin_fmaf(byte_f32<0>(lo), d0, c0), __builtin_fmaf(byte_f32<1>(lo), d0, c0)),
                          pack_bf16(__builtin_fmaf(byte_f32<2>(lo), d0, c0), __builtin_fmaf(byte_f32<3>(lo), d0, c0)),
                          pack_bf16(__builtin_fmaf(byte_f32<0>(hi), d1, c1), __builtin_fmaf(byte_f32<1>(hi), d1, c1)),
                          pack_bf16(__builtin_fmaf(byte_f32<2>(hi), d1, c1), __builtin_fmaf(byte_f32<3>(hi), d1, c1)));
    } else if constexpr (FMT == FMT_MXFP4) {  // the code's doubled value + 12 as an unsigned byte, times the block's power of two: exact in bf16
        const float d = e8m0_half((r.m[0] >> (8 * b)) & 0xFF);
        return dequant_u8x8(mxfp4_values<12>(cw[b] & 0x0F0F0F0Fu), mxfp4_values<12>((cw[b] >> 4) & 0x0F0F0F0Fu), d, -12.0f * d);
    } else if constexpr (FMT == FMT_Q40) {  // the block's own scale: word b / 2, half b % 2; (nib - 8) * d
        const float d = f16_bits_to_f32((uint16_t)((b & 1) ? r.m[b >> 1] >> 16 : r.m[b >> 1] & 0xFFFF));
        return dequant_q4m(cw[b], d, -8.0f * d);
    } else if constexpr (FMT == FMT_Q4M) {
        const int g = b >> 1;
        const float d = f16_bits_to_f32((uint16_t)(g ? r.m[0] >> 16 : r.m[0] & 0xFFFF));
        const float off = bf16_bits_to_f32((uint16_t)(g ? r.m[1] >> 16 : r.m[1] & 0xFFFF));
        return dequant_q4m(cw[b], d, off - 8.0f * d);
    } else if constexpr (q8_format(FMT)) {  // block b = 2 h + e: codes 8 kq .. + 7 of block e of record h; q * d as (q + 128) * d - 128 d
        const int h = b >> 1, e = b & 1;
        float d = FMT == FMT_Q8F ? __uint_as_float(r.m[b]) : f16_bits_to_f32((uint16_t)(e ? r.m[h] >> 16 : r.m[h] & 0xFFFF));
        if (h && 2 * s + 1 >= t8_steps(w.n_in)) d = 0.0f;  // the step's second record lies past the row
        return dequant_u8x8(cw[2 * b] ^ 0x80808080u, cw[2 * b + 1] ^ 0x80808080u, d, -128.0f * d);
    } else if constexpr (k45_format(FMT)) {  // block b = 2 jj + e: the low (e = 0) or high nibbles of the chunk's byte pair jj
        const float d = f16_bits_to_f32((uint16_t)(r.m[2] & 0xFFFF)), dmin = f16_bits_to_f32((uint16_t)(r.m[2] >> 16));
        const int jj = b >> 1, e = b & 1;
        const uint32_t lo = jj ? r.c.z : r.c.x, hi = jj ? r.c.w : r.c.y;
        const float sc = (float)((r.m[0] >> (8 * b)) & 0xFF), mn = (float)((r.m[1] >> (8 * b)) & 0xFF);
        uint32_t w0 = (lo >> (4 * e)) & 0x0F0F0F0Fu, w1 = (hi >> (4 * e)) & 0x0F0F0F0Fu;
        if (FMT == FMT_Q5_K) {  // the fifth bits of the block's two dwords: bits 8 k + 2 b and 8 k + 2 b + 1 of the plane
            w0 |= ((r.c2.x >> (2 * b)) & 0x01010101u) << 4;
            w1 |= ((r.c2.x >> (2 * b + 1)) & 0x01010101u) << 4;
        }
        return dequant_u8x8(w0, w1, d * sc, -(dmin * mn));
    } else if constexpr (FMT == FMT_Q6_K) {  // block b = 2 h + e: codes 8 e .. + 7 of the lane's 16 columns of half h
        const float d = f16_bits_to_f32((uint16_t)(r.m[2] & 0xFFFF));
        const int h = b >> 1, e = b & 1;
        const uint32_t src = e ? (h ? r.c.w : r.c.y) : (h ? r.c.z : r.c.x), hh = (h ? r.c2.y : r.c2.x) >> (4 * e);
        const uint32_t w0 = (src & 0x0F0F0F0Fu) | ((hh & 0x03030303u) << 4);
        const uint32_t w1 = ((src >> 4) & 0x0F0F0F0Fu) | (((hh >> 2) & 0x03030303u) << 4);
        const float dsc = d * (float)(int)(int8_t)((r.m[h] >> (8 * (lane >> 4))) & 0xFF);
        return dequant_u8x8(w0, w1, dsc, -32.0f * dsc);
    } else {  // FP8: bytes 8 b .. 8 b + 7 of the lane's 32; exact in bf16, the block scale multiplies in f32 before the rounding
        const float sc = __uint_as_float(r.m[0]);
        const f32x2 v0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)cw[2 * b], false);
        const f32x2 v1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)cw[2 * b], true);
        const f32x2 v2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)cw[2 * b + 1], false);
        const f32x2 v3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)cw[2 * b + 1], true);
        return make_uint4(pack_bf16(v0.x * sc, v0.y * sc), pack_bf16(v1.x * sc, v1.y * sc), pack_bf16(v2.x * sc, v2.y * sc), pack_bf16(v3.x * sc, v3.y * sc));
    }
}

}  // namespace
}  // namespace oxhip

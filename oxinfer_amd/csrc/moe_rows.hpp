// Rows of activations as the operands of the bf16 grouped expert matmuls (moe_bf16.hip): shared with the routing kernel (moe.hip), which
// makes them beside its own work.
#pragma once
#include "internal.hpp"

namespace oxhip {

// The formats whose records' lane (kq, row) holds eight consecutive columns of a block (Q8_0, Q4_K); the T4M geometry holds four of
// either half.
__host__ __device__ constexpr bool std_columns(int f) { return f == FMT_Q8_0 || f == FMT_Q4_K; }

// Eight columns of a block become an operand's 16 bytes in the order 0, 2, 1, 3, 4, 6, 5, 7: the order in which one mask takes the
// codes' pairs out of a record's dword (moe_bf16_body's `operand`). Also their sum, of the rounded values.
__device__ __forceinline__ uint4 pack_columns(const float* v, float* sum) {
    uint32_t h[8];
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        h[j] = f32_to_bf16_bits(v[j]);
        s += __uint_as_float(h[j] << 16);
    }
    *sum = s;
    return make_uint4(h[0] | (h[2] << 16), h[1] | (h[3] << 16), h[4] | (h[6] << 16), h[5] | (h[7] << 16));
}

// Rows of x as bf16 in the order of the matrix operands, made once per token (its routed copies are gathered from here): 16 bytes
// [row][block of 32][kq] = the row's columns 32 b + {4 kq .. + 3, 16 + 4 kq .. + 3} (STD: 32 b + 8 kq + {0 .. 7}), and the sum of
// every block's rounded values as f32 [row][block]. Unit i of a launch: 16 bytes, four lanes to a block.
template <bool STD>
__device__ __forceinline__ void moe_row_unit(const float* __restrict__ x, size_t i, size_t units, uint4* __restrict__ xb, float* __restrict__ sums) {
    if (i >= units) return;  // (uniform over a block's four lanes)
    const size_t b = i >> 2;
    const uint32_t kq = (uint32_t)i & 3;
    const float4 f0 = *reinterpret_cast<const float4*>(x + 32 * b + (STD ? 8 : 4) * kq), f1 = *reinterpret_cast<const float4*>(x + 32 * b + (STD ? 8 * kq + 4 : 4 * kq + 16));
    const float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    float sum;
    xb[i] = pack_columns(v, &sum);
    sum += dpp_f32<0xB1>(sum);  // quad_perm [1,0,3,2]
    sum += dpp_f32<0x4E>(sum);  // quad_perm [2,3,0,1]
    if (kq == 0) sums[b] = sum;
}

}  // namespace oxhip

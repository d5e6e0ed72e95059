// Arithmetic shared by the int8 weight-only GEMV kernels: the canonical summation order's
// blocking of K, the exact int8 -> packed-bf16 widening and the MFMA steps of a chain.  Every kernel that includes this
// produces the same bits for the same (weight row, activation row).
#pragma once

#include "common.hpp"

namespace cmi {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Segments per unit: the largest of 4,3,2,1 that pads K by at most a fifth.
__host__ __device__ inline int unit_segments(int nseg) {
    for (int u = 4; u > 1; --u) {
        const int padded = (nseg + u - 1) / u * u;
        if ((padded - nseg) * 5 <= padded) return u;
    }
    return 1;
}

// Four int8 in one dword -> two packed-bf16 pairs (k, k+1) and (k+2, k+3).
__device__ __forceinline__ void widen4(uint32_t w, bf16x2_t &lo, bf16x2_t &hi) {
    const float f0 = (float)(int8_t)(w);
    const float f1 = (float)(int8_t)(w >> 8);
    const float f2 = (float)(int8_t)(w >> 16);
    const float f3 = (float)(int8_t)(w >> 24);
    // Integers up to 127 occupy only the upper 16 bits of their fp32 pattern,
    // so taking the high halves is an exact conversion to bf16.
    const uint32_t p0 = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
    const uint32_t p1 = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
    lo = __builtin_bit_cast(bf16x2_t, p0);
    hi = __builtin_bit_cast(bf16x2_t, p1);
}

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));

// Sixteen codes of a weight row as the four MFMA steps take them, four k each.
struct Chunk {
    bf16x4_t step[4];
};

__device__ __forceinline__ bf16x4_t pair_bits(uint32_t lo, uint32_t hi) { return __builtin_bit_cast(bf16x4_t, make_uint2(lo, hi)); }

__device__ __forceinline__ Chunk widen_chunk(const u32x4 &w) {
    Chunk c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        bf16x2_t lo, hi;
        widen4(w[i], lo, hi);
        c.step[i] = pair_bits(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
    }
    return c;
}

// One 16-element chunk of a lane's chain, k ascending: v_mfma_f32_4x4x4_16b_bf16 works on 16 blocks of four lanes; for block b and
// lane 4b + j, register i of v gains the four products of the codes in lane 4b + i with the activations in lane 4b + j.  The products
// are exact; they and what v held are cut off 26 bits below the largest of their exponents, summed, and rounded once (probed on the device).
__device__ __forceinline__ v4f32 chain_chunk(v4f32 v, const Chunk &w, const uint4 &x0, const uint4 &x1) {
    v = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(w.step[0], pair_bits(x0.x, x0.y), v, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(w.step[1], pair_bits(x0.z, x0.w), v, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(w.step[2], pair_bits(x1.x, x1.y), v, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(w.step[3], pair_bits(x1.z, x1.w), v, 0, 0, 0);
    return v;
}

// The chain of the lane's own codes with its own activations: the diagonal of its block.
__device__ __forceinline__ float own_chain(v4f32 v, int lane) {
    const float a = (lane & 1) ? v.y : v.x, b = (lane & 1) ? v.w : v.z;
    return (lane & 2) ? b : a;
}

}  // namespace cmi

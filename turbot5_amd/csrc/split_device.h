// fp32 numbers as sums of three bf16 ones, for fp32 products on the 16-bit matrix cores (gemm_f32.hip, attn_f32.hip).
//
// x = h + m + l: h is x rounded to bf16 (8 significant bits), m the rest rounded, l the rest of that, so the three hold the
// 24 bits of x.  Of the nine products of two such sums the six largest are formed, each with an fp32 accumulator; the three
// left out are at most 2^-24 of the product.  v_mfma_f32_32x32x16_bf16 does sixteen times the multiply-adds of
// v_mfma_f32_32x32x2_f32 per cycle, so six of them take 3/8 of the time.
//
// A part holds multiples of 2^-133 and an fp32 number is one of 2^-149, so kernels split x times kSplitScale = 2^16: its parts
// are exact for every x down to the smallest denormal one (unscaled, numbers below 2^-110 lose bits: 2^-17 of themselves at
// 2^-117).  The scales of a product's operands are taken out of its fp32 sum, exactly.
//
// An infinity, or a value that times 2^16 rounds to one in bf16 (2^112 and more), gives infinity minus infinity in m and l: what fp32
// arithmetic would leave finite or infinite may come out as NaN, and so may a scaled sum past the largest number.  Every such
// case leaves a value in the result that is not finite (h takes part in a product of its own), which is what the kernels test
// before they store, to form the result again in fp32.
#pragma once
#include <hip/hip_runtime.h>

#include "mfma16_device.h"

namespace t5a {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kPlanes = 3;
constexpr float kSplitScale = 0x1p16f, kSplitBack = 0x1p-16f;

// (two values at a time: a packed pair is widened with a shift and a mask)
__device__ __forceinline__ void split3(const f32x8 x, bf16x8 (&out)[kPlanes]) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    u32x4 w[kPlanes];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
        for (int q = 0; q < kPlanes; ++q) {
            w[q][i] = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
            if (q + 1 < kPlanes) {
                a -= __builtin_bit_cast(float, w[q][i] << 16);
                b -= __builtin_bit_cast(float, w[q][i] & 0xffff0000u);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kPlanes; ++q) out[q] = __builtin_bit_cast(bf16x8, w[q]);
}

}  // namespace t5a

// 32-bit numbers as sums of three bfloat16 ones, each what the one before leaves, rounded to the nearest: what lets the bfloat16 matrix cores multiply all 24 bits of
// them (gemm_pieces.h, attention_pieces.h).
#pragma once

#include "common.h"

namespace pieces {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Numbers 2 e and 2 e + 1 of a lane's eight -> their places in three operands of pieces. (A number that the first rounding makes infinite leaves sums that are not finite, as an infinity does.)
__device__ __forceinline__ void split_pair(const i32x4 (&raw)[2], int e, bf16x8 (&out)[3]) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
    const int first = raw[e / 2][e % 2 * 2], second = raw[e / 2][e % 2 * 2 + 1];
    float rest[2] = {__builtin_bit_cast(float, first), __builtin_bit_cast(float, second)};
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const bf16x2 pair = __builtin_convertvector((f32x2{rest[0], rest[1]}), bf16x2);
        out[p][2 * e] = pair[0], out[p][2 * e + 1] = pair[1];
        if (p < 2) {
            const uint32_t bits = __builtin_bit_cast(uint32_t, pair);
            rest[0] -= __builtin_bit_cast(float, bits << 16);
            rest[1] -= __builtin_bit_cast(float, bits & 0xffff0000u);
        }
    }
}

}  // namespace pieces

// f32 values as sums of bf16 terms, for the matrix cores.  Included into one
// anonymous namespace per translation unit.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace accel {
namespace {

typedef __bf16 sp_bf16x2 __attribute__((ext_vector_type(2)));
typedef float sp_f32x2 __attribute__((ext_vector_type(2)));

// Two values as TERMS bf16 pairs (t[0] the largest): each the RNE bf16 of what
// the previous ones leave, the remainder v - term exact in f32.  Three terms
// hold an f32 to 2^-27 of itself; two hold an f16 (11 bits) exactly.  The
// remainder is a widening and a subtraction on the VALU: a v_dot2_f32_bf16 of
// the term against -1 is one instruction less per value, but dot products run
// on the matrix pipe, and four of them beside an MFMA made its slot 29 ns
// where eight VALU instructions make it 20-23 (16 alone; gfx950, one and two
// waves a SIMD).  Where the VALU count and not the matrix pipe sets the time
// (the few-rows decode kernel) the dot product stays: 92.7 against 90.8 us for
// the decode MoE.
template <int TERMS>
__device__ __forceinline__ void split_terms(float v0, float v1, uint32_t (&t)[TERMS]) {
#pragma unroll
    for (int i = 0; i < TERMS; i++) {
        t[i] = __builtin_bit_cast(uint32_t,
                                  __builtin_convertvector((sp_f32x2){v0, v1}, sp_bf16x2));
        if (i + 1 < TERMS) {
            v0 -= __uint_as_float(t[i] << 16);
            v1 -= __uint_as_float(t[i] & 0xffff0000u);
        }
    }
}

}  // namespace
}  // namespace accel

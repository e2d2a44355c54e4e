// mfma.hpp -- bf16 operand helpers shared by the MFMA GEMM kernels.
#pragma once
#include "common.hpp"

namespace atlas {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the high halves of two floats (their bf16 truncations), a low
__device__ __forceinline__ uint32_t bf16_hi2(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// two floats rounded to nearest even, a low
__device__ __forceinline__ uint32_t bf16_rne2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}

// the remainders of two floats' truncations, rounded to nearest even, a low
__device__ __forceinline__ uint32_t bf16_lo2(float a, float b) {
    return bf16_rne2(a - __uint_as_float(__float_as_uint(a) & 0xFFFF0000u),
                     b - __uint_as_float(__float_as_uint(b) & 0xFFFF0000u));
}

// two f32 with <= 8 significant bits -> packed bf16 pair (a low), exact
__device__ __forceinline__ uint32_t pack_f32_pair(float a, float b) { return bf16_hi2(a, b); }

}  // namespace atlas

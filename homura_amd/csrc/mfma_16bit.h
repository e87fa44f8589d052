// The 32 x 32 x 16 matrix instruction of the 16-bit types, by operand type.
#pragma once

namespace homura {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// f16 weights / 4096, for activations' pieces that are held times it (HALF_LOW, row_pieces.h). Exact down to 2^-24; what that leaves out is 2^-27 of
// a row's largest weight, and the pieces it would meet are 2^-11 of their values.
__device__ __forceinline__ bf16x8_t half_low(bf16x8_t w) {
    return __builtin_bit_cast(bf16x8_t, __builtin_bit_cast(f16x8_t, w) * (_Float16)(1.f / 4096.f));
}

// c + a b, the operands' bits being bf16 or (HF) f16
template <bool HF>
__device__ __forceinline__ f32x16_t mfma32(bf16x8_t a, bf16x8_t b, f32x16_t c) {
    if constexpr (HF)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace homura

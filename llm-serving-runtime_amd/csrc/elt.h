// The 16-bit element types of the attention kernels: MFMA forms and fp32 conversions.
#pragma once

#include "common.h"

namespace mx {

// Element type of q, K, V and the output: fp16 (BF16 = false) or bf16 (MX_PA_BF16). Registers
// and memory hold the 16-bit patterns in half vectors either way; only the MFMA forms and the
// fp32 conversions differ. Probabilities enter P.V rounded to the element type, as the
// reference's SDPA path casts its softmax to the query dtype (paged_attention_triton.py:816).
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef short s16x4v __attribute__((ext_vector_type(4)));
template <bool BF16>
struct Elt;
template <>
struct Elt<false> {
    static __device__ __forceinline__ float4v mma32(half8v a, half8v b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float4v mma16(half4v a, half4v b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ _Float16 round(float x) { return (_Float16)x; }
    static __device__ __forceinline__ float widen(_Float16 x) { return (float)x; }
};
template <>
struct Elt<true> {
    static __device__ __forceinline__ float4v mma32(half8v a, half8v b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b),
                                                       c, 0, 0, 0);
    }
    static __device__ __forceinline__ float4v mma16(half4v a, half4v b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4v, a), __builtin_bit_cast(s16x4v, b),
                                                         c, 0, 0, 0);
    }
    static __device__ __forceinline__ _Float16 round(float x) { return __builtin_bit_cast(_Float16, (__bf16)x); }
    static __device__ __forceinline__ float widen(_Float16 x) { return (float)__builtin_bit_cast(__bf16, x); }
};

}  // namespace mx

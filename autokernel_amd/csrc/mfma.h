// mfma.h -- the 16-bit MFMA wrapper shared by the GEMM and attention sources.
#pragma once
#include "ak_common.h"

namespace ak {

// D = A B + C on v_mfma_f32_16x16x32: lane l holds 8 consecutive k (k group l / 16) of row l % 16 of A
// and of column l % 16 of B, and D[4 (l / 16) + v][l % 16] in element v.
template <typename T>
__device__ __forceinline__ f32x4 mfma16x16x32(const u32x4& a, const u32x4& b, const f32x4& c);
template <>
__device__ __forceinline__ f32x4 mfma16x16x32<TF16>(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16x16x32<TBF16>(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace ak

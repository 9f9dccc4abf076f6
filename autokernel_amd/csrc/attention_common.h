// attention_common.h -- what the attention sources share: softmax helpers, and the few-row kernel's
// launcher (attention_rows.hip) for the dispatch in attention.hip.
#pragma once
#include "ak_common.h"

namespace ak {

constexpr float kFaLog2e = 1.4426950408889634f;

template <typename T>
__device__ __forceinline__ uint32_t fa2_pack(float a, float b);
template <>
__device__ __forceinline__ uint32_t fa2_pack<TF16>(float a, float b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, f16x2));
}
template <>
__device__ __forceinline__ uint32_t fa2_pack<TBF16>(float a, float b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, b2));
}
// acc + p.lo + p.hi (p: two packed values)
template <typename T>
__device__ __forceinline__ float fa2_sum2(uint32_t p, float acc);
template <>
__device__ __forceinline__ float fa2_sum2<TF16>(uint32_t p, float acc) {
  const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p), one, acc, false);
}
template <>
__device__ __forceinline__ float fa2_sum2<TBF16>(uint32_t p, float acc) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 one = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, p), one, acc, false);
}
// NaN-propagating max (v_maximum3_f32 / v_maximum_f32). fmaxf would ignore a NaN score, and on
// MFMA results the compiler then quiets each operand first (one v_max_f32 per operand: 11 more
// instructions per 64-key tile). A row whose scores hold a NaN comes out NaN either way: its true
// max fails the overflow test below.
__device__ __forceinline__ float fa2_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// Few query rows per KV head (decode): see attention_rows.hip.
struct FaRowsPlan {
  bool ok;          // the kernel serves this shape
  int64_t splits;   // key slices; > 1 needs a workspace of ws_bytes
  int64_t ws_bytes;
};
FaRowsPlan fa_rows_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D, bool causal);
template <typename T>
int launch_fa_rows(const void* Q, const void* K, const void* V, void* O, int64_t B, int64_t Hq, int64_t Hkv,
                   int64_t Sq, int64_t Sk, int64_t D, const int64_t* qs, const int64_t* ks, const int64_t* vs,
                   const int64_t* os, float sm_scale, float* ws, int64_t ws_bytes, hipStream_t st);

}  // namespace ak

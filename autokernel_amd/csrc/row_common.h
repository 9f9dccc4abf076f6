// row_common.h -- the row-parallel scheme shared by rmsnorm, layernorm, softmax, cross_entropy
// and the last-dim reductions.
//
// A row of `cols` elements is owned by a group of L lanes (L = 8 .. 1024). Each lane loads up to VPT
// 16-byte vectors (vector v = lane_in_group + j * L) into fp32 registers, so the row is read from
// HBM exactly once and written once. Groups narrower than a wave share the wave (several rows per
// wave, segmented butterflies); groups wider than a wave combine their per-wave partials through
// LDS in a fixed order. Rows narrower than a vector or too wide for registers use the looped kernels
// (one 256-thread block per row, scalar loads, two passes).
//
// ANY: rows of any width >= one vector, at any alignment. 16-byte accesses take any alignment here, but
// those that straddle a 16-byte boundary run at a fraction of the rate (cross-entropy f16 [4096, 16385]:
// 43 us with every load straddling, 36 us so), so a row's vectors are the aligned 16-byte pieces of
// memory it covers, except the first and the last, which are moved to start and end with the row.
// The elements that such an end shares with its neighbour are left out of sums at the end (maxima
// take them twice, and both lanes store the same values). Measured, f16, us, against the kernels such
// rows took before (2-byte loads in two or three passes, dword pairs, fp32-cached blocks): layernorm
// [4097, 4097] 46.0 -> 16.8, rmsnorm 27 -> 15, row sums 15.4 -> 8.5; softmax [4096, 50257] 185 -> 157,
// [4096, 20001] 92 -> 62, [16000, 1235] 37 -> 15; cross-entropy fp32 [4096, 20001] 144 -> 58. Rows of
// softmax and cross-entropy just under 65536 columns, whose pieces their lanes cannot hold, leave a few
// elements at the row's start to one lane each (softmax [1024, 65535] 61.4 before, 63.6 with straddling vectors of their own, 57.8 so;
// cross-entropy bf16 [300, 65535] 16.2, 19.5, 16.5).
#pragma once
#include <limits.h>

#include "ak_common.h"

namespace ak {


// Reduction over the L lanes of a segment (L <= 64: every lane ends with the segment result; a
// wider group reduces each of its waves here and combines them in group_combine).
template <int L>
__device__ __forceinline__ float seg_sum(float v) { return seg_reduce<(L < kWave ? L : kWave)>(v, OpAdd()); }
template <int L>
__device__ __forceinline__ float seg_max(float v) { return seg_reduce<(L < kWave ? L : kWave)>(v, OpMax()); }
template <int L>
__device__ __forceinline__ float seg_nan_max(float v) { return seg_reduce<(L < kWave ? L : kWave)>(v, OpNanMax()); }

// Combine per-wave partials of a group of L > 64 lanes (L / 64 waves) through LDS.
// Every wave of the block must call it (it contains barriers). kind: 0 sum, 1 max, 2 nan-max.
template <int L, int KIND>
__device__ __forceinline__ float group_combine(float v, float* red) {
  if constexpr (L <= kWave) {
    return v;
  } else {
    constexpr int G = L / kWave;
    __syncthreads();  // previous readers of red are done
    if (lane_id() == 0) red[wave_id()] = v;
    __syncthreads();
    const int g0 = (wave_id() / G) * G;
    float r = red[g0];
#pragma unroll
    for (int i = 1; i < G; ++i) {
      float o = red[g0 + i];
      if constexpr (KIND == 0) r += o;
      else if constexpr (KIND == 1) r = fmaxf(r, o);
      else r = nan_max(r, o);
    }
    return r;
  }
}

template <int L, int KIND>
__device__ __forceinline__ float group_reduce(float v, float* red) {
  if constexpr (KIND == 0) v = seg_sum<L>(v);
  else if constexpr (KIND == 1) v = seg_max<L>(v);
  else v = seg_nan_max<L>(v);
  return group_combine<L, KIND>(v, red);
}

// Launch geometry of a row-cached kernel with L lanes per row.
template <int L>
struct RowGeom {
  static constexpr int kWPB = (L / kWave) > 4 ? (L / kWave) : 4;  // waves per block
  static constexpr int kThreads = kWPB * kWave;
  static constexpr int kRowsPerBlock = kThreads / L;
  // lane index inside the row group and the block-local group index
  __device__ __forceinline__ static int lane_in_row() { return threadIdx.x % L; }
  __device__ __forceinline__ static int group() { return threadIdx.x / L; }
};

typedef u32x4 u32x4_any __attribute__((aligned(2)));
template <bool ANY>
__device__ __forceinline__ u32x4 ldv(const void* p) {
  if constexpr (ANY) return *reinterpret_cast<const u32x4_any*>(p);
  else return ld16(p);
}
template <bool ANY>
__device__ __forceinline__ void stv(void* p, const u32x4& v) {
  if constexpr (ANY) *reinterpret_cast<u32x4_any*>(p) = v;
  else st16(p, v);
}

// The vectors of a row: vector idx holds elements off(idx) .. off(idx) + kVec - 1 and counts those
// in [lo, hi) of them.
// HEAD: see skew.
template <typename T, bool ANY, bool HEAD = false>
struct RowShape {
  int cols, nvec, skew;  // skew: elements between the aligned address at or before the row and its start
  // most: vectors the row's lanes hold. A row that an end piece would take past it (a width just under
  // the widest one, or under 2^31) takes its vectors from its own start instead, or (HEAD) from the first
  // aligned address after it (skew < 0), which leaves head() elements, fewer than kVec, to the caller.
  __device__ __forceinline__ RowShape(const typename T::S* row, int cols_, bool active, int most = INT_MAX / T::kVec)
      : cols(cols_) {
    skew = ANY ? (int)(((uintptr_t)row & 15u) / sizeof(typename T::S)) : 0;
    if (ANY && count() > most) skew = HEAD ? skew - T::kVec : 0;
    nvec = !active ? 0 : ANY ? count() : cols / T::kVec;
  }
  __device__ __forceinline__ int count() const {
    return (int)(((unsigned)cols + (unsigned)skew + T::kVec - 1) / T::kVec);
  }
  __device__ __forceinline__ int head() const { return max(-skew, 0); }
  __device__ __forceinline__ int off(int idx) const {
    return ANY ? min(max(idx * T::kVec - skew, 0), cols - T::kVec) : idx * T::kVec;
  }
  // fn(element) for the elements of vector idx that count; v holds the vector
  template <typename F>
  __device__ __forceinline__ void each(int idx, const float* v, F fn) const {
    const int first = idx * T::kVec - skew;
    if (!ANY || (first >= 0 && first <= cols - T::kVec)) {
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) fn(v[e]);
    } else {
      const int lo = first < 0 ? 0 : first - (cols - T::kVec), hi = first < 0 ? T::kVec - skew : T::kVec;
#pragma unroll
      for (int e = 0; e < T::kVec; ++e)
        if (e >= lo && e < hi) fn(v[e]);
    }
  }
};

// A row cached in fp32 registers: f[j * kVec + e] is element e of vector lane + j * L (0 past the row).
template <typename T, int L, int VPT, bool ANY = false>
struct RowRegs {
  static constexpr int kE = VPT * T::kVec;
  float f[kE];

  __device__ __forceinline__ static bool valid(int j, int gl, int nvec) { return gl + j * L < nvec; }
  // fn(element) for every element of vector j that counts (the vector must be valid)
  template <bool HEAD, typename F>
  __device__ __forceinline__ void each(int j, int gl, const RowShape<T, ANY, HEAD>& sh, F fn) const {
    sh.each(gl + j * L, f + j * T::kVec, fn);
  }

  template <bool HEAD>
  __device__ __forceinline__ void load(const typename T::S* row, const RowShape<T, ANY, HEAD>& sh, int gl) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int idx = gl + j * L;
      // The zeros are opaque to the compiler: it otherwise loads first and writes constant zeros to the
      // lanes past the row in an else branch, behind a wait for the load that keeps later loads (the
      // weights) from overlapping it (layernorm f16 [14223, 448], 56 vectors for 64 lanes: 7.60 us against 7.25).
      u32x4 v = {0u, 0u, 0u, 0u};
      asm("" : "+v"(v));
      if (idx < sh.nvec) v = ldv<ANY>(row + sh.off(idx));
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) f[j * T::kVec + e] = T::lane_elem(v, e);
    }
  }

  // nt: nontemporal stores (outputs far larger than what a consumer could find in cache)
  template <bool HEAD>
  __device__ __forceinline__ void store(typename T::S* row, const RowShape<T, ANY, HEAD>& sh, int gl, bool nt = false) const {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int idx = gl + j * L;
      if (idx < sh.nvec) {
        u32x4 v;
#pragma unroll
        for (int e = 0; e < T::kVec; ++e) T::set_elem(v, e, f[j * T::kVec + e]);
        if (nt) st16_stream(row + sh.off(idx), v);
        else stv<ANY>(row + sh.off(idx), v);
      }
    }
  }
};

// Host-side choice of (L, VPT) for a row of `nvec` 16-byte vectors: about `want` vectors per lane
// (measured on MI355X, cold cache: rmsnorm f16 4096x4096 15.1 us with 4 per lane against 16.6 us
// with 8; softmax f16 8192x8192 43.8 us against 45.5 us; the last-dim sum prefers 2), at most
// 64 fp32 values per lane and 1024 lanes per row. Returns false when the row does not fit.
struct RowPlan {
  int L;
  int vpt;
};
inline int64_t next_pow2(int64_t v) {
  int64_t p = 1;
  while (p < v) p *= 2;
  return p;
}
inline bool plan_row(int64_t nvec, int kvec, RowPlan* p, int want = 4) {
  const int vmax = 64 / kvec;  // 8 for 2-byte types, 16 for fp32
  if (nvec <= kWave) {         // narrow row: a sub-wave segment, one vector per lane
    p->L = (int)(nvec <= 8 ? 8 : next_pow2(nvec));
    p->vpt = 1;
    return true;
  }
  const int tgt = want < vmax ? want : vmax;
  int64_t L = next_pow2(cdiv(nvec, tgt));
  if (L < kWave) L = kWave;
  if (L > 1024) L = 1024;
  const int64_t vpt = next_pow2(cdiv(nvec, L));
  if (vpt > vmax) return false;
  p->L = (int)L;
  p->vpt = (int)vpt;
  return true;
}

// The plan for `rows` rows of `cols` elements; any: at any alignment (the most vectors a row may cover, or,
// where those do not fit, as many as it needs). None where the rows' lanes pass a grid's work-items (2^22
// rows of 1024 lanes); the kernels of 256 threads per row take four times as many.
inline bool plan_row_cols(int64_t rows, int64_t cols, int kvec, bool any, RowPlan* p, int want = 4) {
  if (cols < kvec) return false;
  const bool fits = !any ? plan_row(cols / kvec, kvec, p, want)
                         : plan_row(cdiv(cols + kvec - 1, kvec), kvec, p, want) || plan_row(cdiv(cols, kvec), kvec, p, want);
  if (!fits) return false;
  const int threads = p->L < 256 ? 256 : p->L;  // per block (RowGeom)
  return grid_fits(cdiv(rows, threads / p->L), threads);
}

}  // namespace ak

// Expand a row-cached kernel launch over aligned rows (ANY false) and rows of any width (ANY true).
#define AK_ANY_SWITCH(any, ...)       \
  if (any) {                          \
    constexpr bool ANY = true;        \
    __VA_ARGS__;                      \
  } else {                            \
    constexpr bool ANY = false;       \
    __VA_ARGS__;                      \
  }

// Expand a row-cached kernel launch over the supported (L, VPT) pairs.
//   AK_ROW_SWITCH(plan, L, VPT, { launch<T, L, VPT>(...); })
#define AK_ROW_CASE(Lv, Vv, ...)                              \
  if (plan.L == Lv && plan.vpt == Vv) {                       \
    constexpr int L = Lv;                                     \
    constexpr int VPT = Vv;                                   \
    if constexpr (VPT * T::kVec <= 64) {                      \
      __VA_ARGS__;                                            \
      handled = true;                                         \
    }                                                         \
  }
#define AK_ROW_SWITCH(...)                                                          \
  do {                                                                           \
    AK_ROW_CASE(8, 1, __VA_ARGS__)                                              \
    else AK_ROW_CASE(16, 1, __VA_ARGS__)                                        \
    else AK_ROW_CASE(32, 1, __VA_ARGS__)                                        \
    else AK_ROW_CASE(64, 1, __VA_ARGS__)                                        \
    else AK_ROW_CASE(64, 2, __VA_ARGS__)                                        \
    else AK_ROW_CASE(64, 4, __VA_ARGS__)                                        \
    else AK_ROW_CASE(64, 8, __VA_ARGS__)                                        \
    else AK_ROW_CASE(64, 16, __VA_ARGS__)                                       \
    else AK_ROW_CASE(128, 2, __VA_ARGS__)                                       \
    else AK_ROW_CASE(128, 4, __VA_ARGS__)                                       \
    else AK_ROW_CASE(128, 8, __VA_ARGS__)                                       \
    else AK_ROW_CASE(128, 16, __VA_ARGS__)                                      \
    else AK_ROW_CASE(256, 2, __VA_ARGS__)                                       \
    else AK_ROW_CASE(256, 4, __VA_ARGS__)                                       \
    else AK_ROW_CASE(256, 8, __VA_ARGS__)                                       \
    else AK_ROW_CASE(256, 16, __VA_ARGS__)                                      \
    else AK_ROW_CASE(512, 2, __VA_ARGS__)                                       \
    else AK_ROW_CASE(512, 4, __VA_ARGS__)                                       \
    else AK_ROW_CASE(512, 8, __VA_ARGS__)                                       \
    else AK_ROW_CASE(512, 16, __VA_ARGS__)                                      \
    else AK_ROW_CASE(1024, 2, __VA_ARGS__)                                      \
    else AK_ROW_CASE(1024, 4, __VA_ARGS__)                                      \
    else AK_ROW_CASE(1024, 8, __VA_ARGS__)                                      \
    else AK_ROW_CASE(1024, 16, __VA_ARGS__)                                     \
  } while (0)

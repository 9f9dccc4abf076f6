// rows.hip -- row-parallel ops on gfx950: rmsnorm, layernorm, softmax, cross_entropy and the
// last-dim reductions. All are HBM-bound: each row is read once into registers (row_common.h)
// and written once; reductions are wave64 butterflies plus a fixed-order LDS combine.
#include <limits.h>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "row_common.h"

namespace ak {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kLoopThreads = 256;
constexpr int kWidestRow = 65536;  // elements of a row cached in registers (1024 lanes of 64)
template <typename T, int L, int VPT, bool ANY>
constexpr bool kWidest = ANY && L * VPT * T::kVec == kWidestRow;
// whether the 16-byte pieces of a row this wide may be more than the widest kernel's lanes hold
template <typename T>
inline bool pieces_pass(int64_t cols) {
  return cdiv(cols + T::kVec - 1, T::kVec) > kWidestRow / T::kVec;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Every wave of a 256-thread block calls this; kind as in group_combine.
template <int KIND>
__device__ __forceinline__ float block_reduce(float v, float* red) {
  return group_reduce<kLoopThreads, KIND>(v, red);
}

// =============================================================================================
// RMSNorm. Op sequence of reference.py:28-29, each a tensor op in x's dtype:
//   sq = x**2; ms = mean(sq); t = ms + eps; rms = sqrt(t); q = x / rms; y = q * weight
// so x*x rounds (and may overflow to inf) in f16 before the fp32-accumulated mean.
// =============================================================================================
// FORM 0: reference.py:28-29, y = (x / sqrt(mean(x^2) + eps)) * w.
// FORM 1: a LLaMA block's module (models/llama_7b.py:28-30), y = x * rsqrt(mean(x^2) + eps) * w,
// where rsqrt's result is itself a tensor rounded to the element type.
template <typename T, int FORM>
struct RmsStats {
  // the factor each x is multiplied by before its rounding
  __device__ __forceinline__ static float scale(float ss, int cols, float eps) {
    const float ms = T::rnd(ss / (float)cols);
    const float t = T::rnd(ms + eps);
    if constexpr (FORM == 0) return 1.0f / T::rnd(sqrtf(t));  // x / rms to within one fp32 ulp
    else return T::rnd(1.0f / sqrtf(t));
  }
};

template <typename T, int L, int VPT, int FORM, bool ANY>
__global__ __launch_bounds__(RowGeom<L>::kThreads) void rmsnorm_rows(
    const typename T::S* __restrict__ x, const typename T::S* __restrict__ w,
    typename T::S* __restrict__ y, int64_t rows, int cols, float eps) {
  using G = RowGeom<L>;
  __shared__ float red[G::kWPB];
  const int gl = G::lane_in_row();
  const int64_t row = (int64_t)blockIdx.x * G::kRowsPerBlock + G::group();
  const bool active = row < rows;
  const RowShape<T, ANY> sh(x + row * cols, cols, active, L * VPT);
  RowRegs<T, L, VPT, ANY> r;
  r.load(x + row * cols, sh, gl);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (!ANY || r.valid(j, gl, sh.nvec)) r.each(j, gl, sh, [&](float v) { ss += T::rnd(v * v); });
  }
  ss = group_reduce<L, 0>(ss, red);
  const float inv = RmsStats<T, FORM>::scale(ss, cols, eps);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int idx = gl + j * L;
    if (idx < sh.nvec) {
      // weights load here, after the reduction (measured faster than issuing them with the row:
      // 14.8 against 15.8 us for f16 4096x4096)
      const int off = sh.off(idx);
      const u32x4 wv = ldv<ANY>(w + off);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < T::kVec; ++e)
        T::set_elem(o, e, T::rnd(r.f[j * T::kVec + e] * inv) * T::lane_elem(wv, e));
      stv<ANY>(y + row * cols + off, o);
    }
  }
}

template <typename T, int FORM>
__global__ __launch_bounds__(kLoopThreads) void rmsnorm_loop(
    const typename T::S* __restrict__ x, const typename T::S* __restrict__ w,
    typename T::S* __restrict__ y, int cols, float eps) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  typename T::S* yr = y + (int64_t)blockIdx.x * cols;
  float ss = 0.f;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) {
    const float v = T::to_f(xr[c]);
    ss += T::rnd(v * v);
  }
  ss = block_reduce<0>(ss, red);
  const float inv = RmsStats<T, FORM>::scale(ss, cols, eps);
  for (int c = threadIdx.x; c < cols; c += kLoopThreads)
    yr[c] = T::from_f(T::rnd(T::to_f(xr[c]) * inv) * T::to_f(w[c]));
}

template <typename T, int FORM>
static int launch_rmsnorm(const void* x, const void* w, void* y, int64_t rows, int64_t cols,
                          float eps, hipStream_t s) {
  using S = typename T::S;
  const S* xp = (const S*)x;
  const S* wp = (const S*)w;
  S* yp = (S*)y;
  RowPlan plan;
  const bool any = cols % T::kVec != 0 || !host_aligned16(x) || !host_aligned16(y) || !host_aligned16(w);
  bool handled = false;
  if (plan_row_cols(rows, cols, T::kVec, any, &plan)) {
    AK_ANY_SWITCH(any, AK_ROW_SWITCH({
      const dim3 grid((unsigned)cdiv(rows, RowGeom<L>::kRowsPerBlock));
      rmsnorm_rows<T, L, VPT, FORM, ANY><<<grid, RowGeom<L>::kThreads, 0, s>>>(xp, wp, yp, rows, (int)cols, eps);
    }));
  }
  if (!handled) rmsnorm_loop<T, FORM><<<(unsigned)rows, kLoopThreads, 0, s>>>(xp, wp, yp, (int)cols, eps);
  return record_launch();
}

// =============================================================================================
// LayerNorm: F.layer_norm over the last dim (reference.py:20-23): fp32 mean and biased variance,
// rstd = rsqrt(var + eps), y = (x - mean) * rstd * w + b rounded once.
// =============================================================================================
template <typename T>
__device__ __forceinline__ float ln_out(float v, float mean, float rstd, const typename T::S* w,
                                        const typename T::S* b, int64_t c) {
  float o = (v - mean) * rstd;
  if (w) o *= T::to_f(w[c]);
  if (b) o += T::to_f(b[c]);
  return o;
}

template <typename T, int L, int VPT, bool ANY>
__global__ __launch_bounds__(RowGeom<L>::kThreads) void layernorm_rows(
    const typename T::S* __restrict__ x, const typename T::S* __restrict__ w,
    const typename T::S* __restrict__ b, typename T::S* __restrict__ y, int64_t rows, int cols,
    float eps) {
  using G = RowGeom<L>;
  using R = RowRegs<T, L, VPT, ANY>;
  // With rows of any alignment and on blocks of 1024 lanes, of which a CU holds one or two, the affine
  // parameters load after the reductions, otherwise with the row (us, after / with the row: f16 [4096, 16385]
  // 74 / 99, aligned f16 [1024, 32768] 26.6 / 31.1, fp32 [2048, 16384] 49.8 / 55.4, bf16 [1024, 65536] 58 / 148,
  // whose 64 values a lane spill beside the parameters; but f16 [4096, 4096] 15.5 / 13.7, fp32 [4096, 4096]
  // 24.2 / 20.5).
  constexpr bool kAfter = ANY || L == 1024;
  __shared__ float red[G::kWPB];
  const int gl = G::lane_in_row();
  const int64_t row = (int64_t)blockIdx.x * G::kRowsPerBlock + G::group();
  const bool active = row < rows;
  const RowShape<T, ANY> sh(x + row * cols, cols, active, L * VPT);
  const int nvec = sh.nvec;
  R r;
  r.load(x + row * cols, sh, gl);
  u32x4 wv[VPT], bv[VPT];
  auto affine = [&](int j) {
    const int idx = gl + j * L;
    wv[j] = (w && idx < nvec) ? ldv<ANY>(w + sh.off(idx)) : u32x4{0u, 0u, 0u, 0u};
    bv[j] = (b && idx < nvec) ? ldv<ANY>(b + sh.off(idx)) : u32x4{0u, 0u, 0u, 0u};
  };
  if constexpr (!kAfter) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) affine(j);
  }
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (!ANY || R::valid(j, gl, nvec)) r.each(j, gl, sh, [&](float v) { s += v; });  // past the row: zeros
  }
  const float mean = group_reduce<L, 0>(s, red) / (float)cols;
  float d = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (R::valid(j, gl, nvec))
      r.each(j, gl, sh, [&](float v) {
        const float t = v - mean;
        d += t * t;
      });
  }
  const float var = group_reduce<L, 0>(d, red) / (float)cols;
  const float rstd = rsqrtf(var + eps);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int idx = gl + j * L;
    if (idx < nvec) {
      if constexpr (kAfter) affine(j);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) {
        float v = (r.f[j * T::kVec + e] - mean) * rstd;
        if (w) v *= T::lane_elem(wv[j], e);
        if (b) v += T::lane_elem(bv[j], e);
        T::set_elem(o, e, v);
      }
      stv<ANY>(y + row * cols + sh.off(idx), o);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kLoopThreads) void layernorm_loop(
    const typename T::S* __restrict__ x, const typename T::S* __restrict__ w,
    const typename T::S* __restrict__ b, typename T::S* __restrict__ y, int cols, float eps) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  typename T::S* yr = y + (int64_t)blockIdx.x * cols;
  float s = 0.f;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) s += T::to_f(xr[c]);
  const float mean = block_reduce<0>(s, red) / (float)cols;
  float d = 0.f;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) {
    const float t = T::to_f(xr[c]) - mean;
    d += t * t;
  }
  const float rstd = rsqrtf(block_reduce<0>(d, red) / (float)cols + eps);
  for (int c = threadIdx.x; c < cols; c += kLoopThreads)
    yr[c] = T::from_f(ln_out<T>(T::to_f(xr[c]), mean, rstd, w, b, c));
}

template <typename T>
static int launch_layernorm(const void* x, const void* w, const void* b, void* y, int64_t rows,
                            int64_t cols, float eps, hipStream_t s) {
  using S = typename T::S;
  const S* xp = (const S*)x;
  const S* wp = (const S*)w;
  const S* bp = (const S*)b;
  S* yp = (S*)y;
  RowPlan plan;
  const bool any = cols % T::kVec != 0 || !host_aligned16(x) || !host_aligned16(y) ||
                   (w && !host_aligned16(w)) || (b && !host_aligned16(b));
  bool handled = false;
  if (plan_row_cols(rows, cols, T::kVec, any, &plan)) {
    AK_ANY_SWITCH(any, AK_ROW_SWITCH({
      const dim3 grid((unsigned)cdiv(rows, RowGeom<L>::kRowsPerBlock));
      layernorm_rows<T, L, VPT, ANY><<<grid, RowGeom<L>::kThreads, 0, s>>>(xp, wp, bp, yp, rows, (int)cols, eps);
    }));
  }
  if (!handled) layernorm_loop<T><<<(unsigned)rows, kLoopThreads, 0, s>>>(xp, wp, bp, yp, (int)cols, eps);
  return record_launch();
}

// =============================================================================================
// Softmax over the last dim (reference.py:15-17): fp32 max, exp and sum, one rounding.
// =============================================================================================
// HEAD (also of ce_rows): unaligned rows of a width whose pieces may pass what the lanes hold; the others do
// without the elements it leaves at the row's start (softmax f16 [4096, 50257] 158.9 us with them, 156.3).
template <typename T, int L, int VPT, bool ANY, bool HEAD>
__global__ __launch_bounds__(RowGeom<L>::kThreads) void softmax_rows(
    const typename T::S* __restrict__ x, typename T::S* __restrict__ y, int64_t rows, int cols, int nt_out) {
  using G = RowGeom<L>;
  using R = RowRegs<T, L, VPT, ANY>;
  __shared__ float red[G::kWPB];
  const int gl = G::lane_in_row();
  const int64_t row = (int64_t)blockIdx.x * G::kRowsPerBlock + G::group();
  const bool active = row < rows;
  const RowShape<T, ANY, HEAD> sh(x + row * cols, cols, active, L * VPT);
  const bool has_head = HEAD && gl < sh.head();
  R r;
  r.load(x + row * cols, sh, gl);
  float h = has_head ? T::to_f(x[row * cols + gl]) : -INFINITY, m = h;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (R::valid(j, gl, sh.nvec))
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) m = fmaxf(m, r.f[j * T::kVec + e]);
  m = group_reduce<L, 1>(m, red);
  const float mb = m * kLog2e;
  float s = 0.f;
  if (has_head) s = h = fast_exp2(__builtin_fmaf(h, kLog2e, -mb));
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (R::valid(j, gl, sh.nvec)) {
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) r.f[j * T::kVec + e] = fast_exp2(__builtin_fmaf(r.f[j * T::kVec + e], kLog2e, -mb));
      r.each(j, gl, sh, [&](float p) { s += p; });
    }
  }
  s = group_reduce<L, 0>(s, red);
  const float inv = 1.0f / s;
#pragma unroll
  for (int e = 0; e < R::kE; ++e) r.f[e] *= inv;
  r.store(y + row * cols, sh, gl, nt_out != 0);
  if (has_head) y[row * cols + gl] = T::from_f(h * inv);
}

// Online (max, sum-of-exp) accumulator used by the looped softmax and cross-entropy kernels.
// -inf entries contribute nothing, +inf or NaN entries make the sum NaN (torch's softmax result).
struct OnlineMS {
  float m = -INFINITY;
  float s = 0.f;
  bool nan = false;
  __device__ __forceinline__ void add(float v) {
    if (v != v) { nan = true; return; }
    const float mn = fmaxf(m, v);
    if (mn == -INFINITY) return;
    s = s * fast_exp2((m - mn) * kLog2e) + fast_exp2((v - mn) * kLog2e);
    m = mn;
  }
};

// Combine per-thread (m, s) over a 256-thread block in fixed order; returns the row's (M, S).
__device__ __forceinline__ void block_combine_ms(OnlineMS a, float* red, float* M, float* S) {
  float mx = block_reduce<1>(a.m, red);
  float sc = (a.m == -INFINITY) ? 0.f : a.s * fast_exp2((a.m - mx) * kLog2e);
  if (a.nan) sc = NAN;
  float tot = block_reduce<0>(sc, red);
  *M = mx;
  *S = tot;
}

// Streaming row statistics (softmax_stream, ce_stream): one row per 256-thread block, read once as the
// aligned 16-byte vectors it covers (row_common.h, ANY) with an online (max, sum) per thread and
// kStreamUnroll vectors in flight. Nothing is cached in registers, so up to eight rows are in flight
// per CU. Per chunk: the chunk max (NaN-propagating), one rescale of the running sum, then
// exp2((x - max) log2 e) per element; the per-thread (max, sum) pairs combine in a fixed order
// (block_combine_ms), as in the looped kernels.
constexpr int kStreamUnroll = 4;
template <typename T>
__device__ __forceinline__ void stream_ms(const typename T::S* xr, int cols, float* red, float* M, float* S) {
  const RowShape<T, true> sh(xr, cols, true);
  float m = -INFINITY, s = 0.f;
  for (int b = threadIdx.x; b < sh.nvec; b += kLoopThreads * kStreamUnroll) {
    u32x4 p[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u)  // past the row: its last vector, left out of the sum
      p[u] = ldv<true>(xr + sh.off(min(b + u * kLoopThreads, sh.nvec - 1)));
    float cm = -INFINITY;
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u)
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) cm = __builtin_elementwise_maximum(cm, T::lane_elem(p[u], e));
    const float mn = __builtin_elementwise_maximum(m, cm);
    if (mn == -INFINITY) continue;  // nothing but -inf so far
    s = (m == -INFINITY) ? 0.f : s * fast_exp2((m - mn) * kLog2e);
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u)
      if (b + u * kLoopThreads < sh.nvec) {
        float v[T::kVec];
#pragma unroll
        for (int e = 0; e < T::kVec; ++e) v[e] = T::lane_elem(p[u], e);
        sh.each(b + u * kLoopThreads, v, [&](float x) { s += fast_exp2((x - mn) * kLog2e); });
      }
    m = mn;
  }
  OnlineMS a;
  a.m = m;
  a.s = s;
  a.nan = (m != m);
  block_combine_ms(a, red, M, S);
}

// Streaming softmax: the online pass above, then a second read of the row (from the caches when they
// still hold it) that writes exp2((x - M) log2 e) / S. The write pass takes the row's whole aligned vectors
// and the few elements at its ends one by one, so that no lane reads what another writes: y may be x.
template <typename T>
__global__ __launch_bounds__(kLoopThreads) void softmax_stream(const typename T::S* __restrict__ x,
                                                               typename T::S* __restrict__ y, int cols) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  typename T::S* yr = y + (int64_t)blockIdx.x * cols;
  float M, S;
  stream_ms<T>(xr, cols, red, &M, &S);
  const float inv = 1.0f / S;
  auto value = [&](float v) { return fast_exp2((v - M) * kLog2e) * inv; };
  const int skew = RowShape<T, true>(xr, cols, true).skew, head = skew ? T::kVec - skew : 0;
  const int nvec = (cols - head) / T::kVec, tail = head + nvec * T::kVec;
  const typename T::S* xv = xr + head;
  typename T::S* yv = yr + head;
  for (int b = threadIdx.x; b < nvec; b += kLoopThreads * kStreamUnroll) {
    u32x4 p[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u)
      p[u] = ldv<true>(xv + min(b + u * kLoopThreads, nvec - 1) * T::kVec);
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u)
      if (b + u * kLoopThreads < nvec) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < T::kVec; ++e) T::set_elem(o, e, value(T::lane_elem(p[u], e)));
        stv<true>(yv + (b + u * kLoopThreads) * T::kVec, o);
      }
  }
  // one lane per element: the first ones take the head, the next ones the tail (fewer than kVec each)
  const int t = threadIdx.x, past = t - head;
  if (t < head) yr[t] = T::from_f(value(T::to_f(xr[t])));
  else if (past < cols - tail) yr[tail + past] = T::from_f(value(T::to_f(xr[tail + past])));
}

template <typename T>
__global__ __launch_bounds__(kLoopThreads) void softmax_loop(
    const typename T::S* __restrict__ x, typename T::S* __restrict__ y, int cols) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  typename T::S* yr = y + (int64_t)blockIdx.x * cols;
  OnlineMS a;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) a.add(T::to_f(xr[c]));
  float M, S;
  block_combine_ms(a, red, &M, &S);
  // The write pass uses the online pass's exponent form, (x - M) log2 e. The fused form
  // x log2 e - round(M log2 e) of the cached kernels would shift every exponent by the rounding of
  // M log2 e (0.008 at |M| ~ 1e5), a scale that S, summed in the other form, does not share.
  const float inv = 1.0f / S;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads)
    yr[c] = T::from_f(fast_exp2((T::to_f(xr[c]) - M) * kLog2e) * inv);
}

template <typename T>
static int launch_softmax(const void* x, void* y, int64_t rows, int64_t cols, hipStream_t s) {
  using S = typename T::S;
  const S* xp = (const S*)x;
  S* yp = (S*)y;
  RowPlan plan;
  bool handled = false;
  // An output larger than the 256 MB Infinity Cache is stored nontemporally; smaller outputs keep
  // plain stores, so the consumer that usually reads them next finds them in cache. Measured, f16
  // [8192, 8192] (128 MiB), cold, softmax then a consumer of its output: with a reduce sum 62.9 us
  // plain against 69.7 us nontemporal, with a [8192, 8192] x [8192, 128] product 88.2 against
  // 89.5 us. Nontemporal stores win only for back-to-back softmax calls whose outputs nobody reads
  // (the dirty lines' write-back then lands in the next kernel): 56.3 against 67.3 us per
  // RoPE(q), RoPE(k), softmax step.
  const int nt_out = rows * cols * (int64_t)sizeof(S) > ((int64_t)256 << 20);
  const bool any = cols % T::kVec != 0 || !host_aligned16(x) || !host_aligned16(y);
  if (plan_row_cols(rows, cols, T::kVec, any, &plan)) {
    AK_ANY_SWITCH(any, AK_ROW_SWITCH({
      const dim3 grid((unsigned)cdiv(rows, RowGeom<L>::kRowsPerBlock));
      auto run = [&](auto kernel) { launch_timed(kernel, grid, dim3(RowGeom<L>::kThreads), 0, s, xp, yp, rows, (int)cols, nt_out); };
      if (kWidest<T, L, VPT, ANY> && pieces_pass<T>(cols)) run(softmax_rows<T, L, VPT, ANY, kWidest<T, L, VPT, ANY>>);
      else run(softmax_rows<T, L, VPT, ANY, false>);
    }));
  } else if (cols >= T::kVec) {
    launch_timed(softmax_stream<T>, dim3((unsigned)rows), dim3(kLoopThreads), 0, s, xp, yp, (int)cols);
    handled = true;
  }
  if (!handled) launch_timed(softmax_loop<T>, dim3((unsigned)rows), dim3(kLoopThreads), 0, s, xp, yp, (int)cols);
  return record_launch();
}

// =============================================================================================
// Cross entropy (reference.py:58-60 = F.cross_entropy, mean reduction, ignore_index):
//   log_softmax in fp32 rounded to the logits' dtype, nll = -logp[target], then the mean of the
//   rounded values accumulated in fp32 and rounded once. Per-row losses go to a caller-owned
//   fp32 workspace; a single-block kernel then reduces them in a fixed order.
// =============================================================================================
template <typename T>
__device__ __forceinline__ float ce_row_loss(const typename T::S* xr, int64_t t, int64_t vocab,
                                             int64_t ignore_index, float M, float S) {
  if (t == ignore_index) return 0.f;
  if (t < 0 || t >= vocab) return NAN;
  const float lp = T::rnd(T::to_f(xr[t]) - M - logf(S));
  return -lp;
}

// The same loss for a sum taken as s = sum 2^(x log2 e - mb), mb = round(M log2 e): the target's
// exponent is formed the same way, so the rounding of mb (a factor 2^-eps in s) cancels in
// lp = (x_t log2 e - mb) ln 2 - log s. Subtracting M directly would leave eps ln 2 in the loss
// (5e-3 at |M| ~ 1e5).
template <typename T>
__device__ __forceinline__ float ce_row_loss_b2(const typename T::S* xr, int64_t t, int64_t vocab,
                                                int64_t ignore_index, float mb, float s) {
  if (t == ignore_index) return 0.f;
  if (t < 0 || t >= vocab) return NAN;
  const float lp = T::rnd(__builtin_fmaf(T::to_f(xr[t]), kLog2e, -mb) * kLn2 - logf(s));
  return -lp;
}

template <typename T, int L, int VPT, bool ANY, bool HEAD>
__global__ __launch_bounds__(RowGeom<L>::kThreads) void ce_rows(
    const typename T::S* __restrict__ x, const int64_t* __restrict__ tgt, float* __restrict__ loss,
    int64_t rows, int cols, int64_t ignore_index) {
  using G = RowGeom<L>;
  using R = RowRegs<T, L, VPT, ANY>;
  __shared__ float red[G::kWPB];
  const int gl = G::lane_in_row();
  const int64_t row = (int64_t)blockIdx.x * G::kRowsPerBlock + G::group();
  const bool active = row < rows;
  const RowShape<T, ANY, HEAD> sh(x + row * cols, cols, active, L * VPT);
  const bool has_head = HEAD && gl < sh.head();
  R r;
  r.load(x + row * cols, sh, gl);
  const float h = has_head ? T::to_f(x[row * cols + gl]) : -INFINITY;
  float m = h;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (R::valid(j, gl, sh.nvec))
#pragma unroll
      for (int e = 0; e < T::kVec; ++e) m = fmaxf(m, r.f[j * T::kVec + e]);
  m = group_reduce<L, 1>(m, red);
  const float mb = m * kLog2e;
  float s = has_head ? fast_exp2(__builtin_fmaf(h, kLog2e, -mb)) : 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (R::valid(j, gl, sh.nvec)) r.each(j, gl, sh, [&](float v) { s += fast_exp2(__builtin_fmaf(v, kLog2e, -mb)); });
  s = group_reduce<L, 0>(s, red);
  if (active && gl == 0) loss[row] = ce_row_loss_b2<T>(x + row * cols, tgt[row], cols, ignore_index, mb, s);
}

// Cross-entropy of a row from the streaming statistics: loss = x_t - M - log S, as in ce_loop.
template <typename T>
__global__ __launch_bounds__(kLoopThreads) void ce_stream(const typename T::S* __restrict__ x,
                                                          const int64_t* __restrict__ tgt,
                                                          float* __restrict__ loss, int cols,
                                                          int64_t ignore_index) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  float M, S;
  stream_ms<T>(xr, cols, red, &M, &S);
  if (threadIdx.x == 0) loss[blockIdx.x] = ce_row_loss<T>(xr, tgt[blockIdx.x], cols, ignore_index, M, S);
}

template <typename T>
__global__ __launch_bounds__(kLoopThreads) void ce_loop(
    const typename T::S* __restrict__ x, const int64_t* __restrict__ tgt, float* __restrict__ loss,
    int cols, int64_t ignore_index) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  OnlineMS a;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) a.add(T::to_f(xr[c]));
  float M, S;
  block_combine_ms(a, red, &M, &S);
  if (threadIdx.x == 0) loss[blockIdx.x] = ce_row_loss<T>(xr, tgt[blockIdx.x], cols, ignore_index, M, S);
}

constexpr int kMeanThreads = 1024;

template <typename T>
__global__ __launch_bounds__(kMeanThreads) void ce_mean(const float* __restrict__ loss,
                                                        const int64_t* __restrict__ tgt,
                                                        typename T::S* __restrict__ out,
                                                        int64_t rows, int64_t ignore_index) {
  __shared__ float red[kMeanThreads / kWave];
  // Thread t adds rows t, t + 1024, t + 2048, ... in that order. Each pass loads eight rows' target
  // and loss before adding any of them, so the loads overlap (a dependent load per row took 4.2 us
  // for 4096 rows); the order of the additions is the same either way.
  constexpr int U = 8;
  float s = 0.f, n = 0.f;
  for (int64_t r0 = threadIdx.x; r0 < rows; r0 += (int64_t)U * kMeanThreads) {
    int64_t t[U];
    float l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = r0 + (int64_t)u * kMeanThreads;
      t[u] = r < rows ? tgt[r] : ignore_index;
      l[u] = r < rows ? loss[r] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (t[u] != ignore_index) {
        s += l[u];
        n += 1.f;
      }
  }
  s = group_reduce<kMeanThreads, 0>(s, red);
  n = group_reduce<kMeanThreads, 0>(n, red);
  if (threadIdx.x == 0) out[0] = T::from_f(s / n);
}

template <typename T>
static int launch_ce(const void* logits, const int64_t* tgt, float* loss, void* out, int64_t rows,
                     int64_t vocab, int64_t ignore_index, hipStream_t s) {
  using S = typename T::S;
  const S* xp = (const S*)logits;
  RowPlan plan;
  const bool any = vocab % T::kVec != 0 || !host_aligned16(logits);
  bool handled = rows == 0;  // no rows: only the mean kernel runs (0 / 0 = NaN, as torch gives)
  const bool planned = plan_row_cols(rows, vocab, T::kVec, any, &plan);
  // 16-bit rows past 32768 columns, and unaligned ones past 16384, stream once the rows fill the chip: a
  // register-cached block of theirs leaves room for one row per CU (us, ce_rows / ce_stream, f16: 4096 x
  // 50264 98 / 81, 4096 x 32769 78 / 56, 4096 x 16385 36 / 30; but 100 x 65536 9.0 / 12.4, aligned 4096 x
  // 32000 49.0 / 54.7, fp32 4096 x 16385 50 / 53).
  const bool stream = sizeof(S) == 2 && rows > 512 && (vocab > 32768 || (any && vocab > 16384));
  if (!handled && planned && !stream) {
    AK_ANY_SWITCH(any, AK_ROW_SWITCH({
      const dim3 grid((unsigned)cdiv(rows, RowGeom<L>::kRowsPerBlock));
      if (kWidest<T, L, VPT, ANY> && pieces_pass<T>(vocab))
        ce_rows<T, L, VPT, ANY, kWidest<T, L, VPT, ANY>><<<grid, RowGeom<L>::kThreads, 0, s>>>(xp, tgt, loss, rows, (int)vocab, ignore_index);
      else
        ce_rows<T, L, VPT, ANY, false><<<grid, RowGeom<L>::kThreads, 0, s>>>(xp, tgt, loss, rows, (int)vocab, ignore_index);
    }));
  } else if (!handled && vocab >= T::kVec) {
    ce_stream<T><<<(unsigned)rows, kLoopThreads, 0, s>>>(xp, tgt, loss, (int)vocab, ignore_index);
    handled = true;
  }
  if (!handled) ce_loop<T><<<(unsigned)rows, kLoopThreads, 0, s>>>(xp, tgt, loss, (int)vocab, ignore_index);
  ce_mean<T><<<1, kMeanThreads, 0, s>>>(loss, tgt, (S*)out, rows, ignore_index);
  return record_launch();
}

// =============================================================================================
// Last-dim reductions (reduce over a contiguous row): sum with fp32 accumulation rounded once
// (x.sum(-1), reference.py:72-74), max exact with NaN propagation (x.max(-1).values, :76-78).
// =============================================================================================
template <typename T, int L, int VPT, bool MAX, bool ANY>
__global__ __launch_bounds__(RowGeom<L>::kThreads) void reduce_rows(
    const typename T::S* __restrict__ x, typename T::S* __restrict__ y, int64_t rows, int cols) {
  using G = RowGeom<L>;
  using R = RowRegs<T, L, VPT, ANY>;
  __shared__ float red[G::kWPB];
  const int gl = G::lane_in_row();
  const int64_t row = (int64_t)blockIdx.x * G::kRowsPerBlock + G::group();
  const bool active = row < rows;
  const RowShape<T, ANY> sh(x + row * cols, cols, active, L * VPT);
  R r;
  r.load(x + row * cols, sh, gl);
  float a = MAX ? -INFINITY : 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (R::valid(j, gl, sh.nvec)) r.each(j, gl, sh, [&](float v) { a = MAX ? nan_max(a, v) : a + v; });
  a = group_reduce<L, MAX ? 2 : 0>(a, red);
  if (active && gl == 0) y[row] = T::from_f(a);
}

template <typename T, bool MAX>
__global__ __launch_bounds__(kLoopThreads) void reduce_loop(const typename T::S* __restrict__ x,
                                                            typename T::S* __restrict__ y, int cols) {
  __shared__ float red[kLoopThreads / kWave];
  const typename T::S* xr = x + (int64_t)blockIdx.x * cols;
  float a = MAX ? -INFINITY : 0.f;
  for (int c = threadIdx.x; c < cols; c += kLoopThreads) {
    const float v = T::to_f(xr[c]);
    a = MAX ? nan_max(a, v) : a + v;
  }
  a = block_reduce<MAX ? 2 : 0>(a, red);
  if (threadIdx.x == 0) y[blockIdx.x] = T::from_f(a);
}

// Reduction over a strided middle dim, x viewed as [outer, reduce, inner]: many short sums. One
// thread per (outer, inner) output; consecutive threads read consecutive inner elements.
template <typename T, bool MAX>
__global__ __launch_bounds__(256) void reduce_cols_short(const typename T::S* __restrict__ x,
                                                         typename T::S* __restrict__ y, int64_t outer,
                                                         int64_t red_n, int64_t inner) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= outer * inner) return;
  const int64_t o = i / inner, c = i % inner;
  const typename T::S* p = x + o * red_n * inner + c;
  float a = MAX ? -INFINITY : 0.f;
  for (int64_t r = 0; r < red_n; ++r) {
    const float v = T::to_f(p[r * inner]);
    a = MAX ? nan_max(a, v) : a + v;
  }
  y[i] = T::from_f(a);
}

// Reduction over a strided middle dim, every other shape. HBM-bound: x is read once. A 256-thread
// block owns CG column groups of V elements (one 16-byte load each; V = 1 when inner is narrower
// than a vector) of one outer index and a slice of the rows; thread (c, r) adds rows r, r + RG, ...
// of its group in fp32, eight loads in flight, and the RG partial sums of a group combine in a
// fixed order through LDS. Where outer and inner alone give too few blocks the rows are cut into
// `slices` (grid y), whose fp32 partials go to a workspace [slices][outer][inner] and are summed by
// a second launch of this kernel (S = TF32 in, T out) in a fixed order: deterministic either way.
// A thread's group may start at any element (rows of an odd inner are not 16-byte aligned; global
// loads take any alignment); the last group is moved back to end at the row's end, so it overlaps
// its neighbour and both write the same values.
// Measured on the sum over dim 0 of bf16 [8192, 4096] (67 MB): one thread per output, 16 blocks in
// all, took 1895 us (35 GB/s); this takes 14.7 us (4.6 TB/s, both launches).
constexpr int kColThreads = 256;
constexpr int kColUnroll = 8;

template <typename S>
struct VecAny;  // 16 bytes at element alignment
template <>
struct VecAny<uint16_t> {
  typedef u32x4 V __attribute__((aligned(2)));
};
template <>
struct VecAny<float> {
  typedef u32x4 V __attribute__((aligned(4)));
};

template <typename T, typename TO, int V, bool MAX>
__global__ __launch_bounds__(kColThreads) void reduce_cols(const typename T::S* __restrict__ x,
                                                           typename TO::S* __restrict__ y,
                                                           float* __restrict__ part, int64_t red_n, int64_t inner,
                                                           int cg_log2, int col_blocks, int64_t slice_rows) {
  static_assert(V == 1 || V == T::kVec, "one element or one 16-byte vector");
  using S = typename T::S;
  __shared__ float lds[kColThreads * V];
  const int CG = 1 << cg_log2, RG = kColThreads >> cg_log2;
  const int c = threadIdx.x & (CG - 1), r = threadIdx.x >> cg_log2;
  const int64_t o = blockIdx.x / (unsigned)col_blocks;
  const int64_t first = ((int64_t)(blockIdx.x % (unsigned)col_blocks) * CG + c) * V;  // before the move back
  const int64_t col = min(first, inner - V);
  const int64_t r0 = blockIdx.y * slice_rows, r1 = min(red_n, r0 + slice_rows);
  float a[V];
#pragma unroll
  for (int e = 0; e < V; ++e) a[e] = MAX ? -INFINITY : 0.f;
  if (first < inner) {
    const S* p = x + (o * red_n + r0 + r) * inner + col;
    const int64_t step = (int64_t)RG * inner;
    auto add = [&](const u32x4& v) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float f = T::lane_elem(v, e);
        a[e] = MAX ? nan_max(a[e], f) : a[e] + f;
      }
    };
    auto ld = [&](const S* q) -> u32x4 {
      if constexpr (V > 1) return *reinterpret_cast<const typename VecAny<S>::V*>(q);
      else if constexpr (sizeof(S) == 2) return u32x4{(uint32_t)*q, 0u, 0u, 0u};
      else return u32x4{__builtin_bit_cast(uint32_t, *q), 0u, 0u, 0u};
    };
    int64_t n = r0 + r < r1 ? (r1 - r0 - r + RG - 1) >> (8 - cg_log2) : 0;  // rows of this thread
    for (; n >= kColUnroll; n -= kColUnroll, p += kColUnroll * step) {
      u32x4 v[kColUnroll];
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u) v[u] = ld(p + u * step);
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u) add(v[u]);
    }
    for (; n > 0; --n, p += step) add(ld(p));
  }
  // RG partials of each column, added pairwise in a fixed tree (element-major: conflict-free)
#pragma unroll
  for (int e = 0; e < V; ++e) lds[e * kColThreads + threadIdx.x] = a[e];
  for (int h = RG >> 1; h > 0; h >>= 1) {
    __syncthreads();
    if (r < h) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        float* q = &lds[e * kColThreads + threadIdx.x];
        const float b = q[h << cg_log2];
        *q = MAX ? nan_max(*q, b) : *q + b;
      }
    }
  }
  if (r != 0 || first >= inner) return;
  if (part) {
    float* q = part + ((int64_t)blockIdx.y * (gridDim.x / (unsigned)col_blocks) + o) * inner + col;
#pragma unroll
    for (int e = 0; e < V; ++e) q[e] = lds[e * kColThreads + threadIdx.x];
  } else {
    typename TO::S* q = y + o * inner + col;
#pragma unroll
    for (int e = 0; e < V; ++e) q[e] = TO::from_f(lds[e * kColThreads + threadIdx.x]);
  }
}

// Launch geometry of reduce_cols.
struct ColPlan {
  bool short_rows;  // reduce_cols_short instead
  bool vec;
  int cg_log2;
  int64_t col_blocks, slices, slice_rows;
};

static ColPlan plan_cols(int64_t outer, int64_t red_n, int64_t inner, int kvec) {
  ColPlan p{};
  // Blocks of the column kernel would be nearly empty, and one thread per output already fills the chip; or
  // the call is small and one thread adds its few rows before a block has combined its row groups (us, one
  // thread per output / column blocks: f16 [2, 300000] 2.8 / 5.0, [8, 300000] 3.4 / 5.0, [16, 262144] 4.1 /
  // 4.7, [3, 542] 2.6 / 3.1, fp32 [2, 1000000] 4.5 / 5.2; but [13, 262144] 6.0 / 5.1, [16, 16384] 3.7 / 3.1,
  // f16 [8, 1000000] 8.1 / 7.0).
  p.short_rows = (red_n * inner < 4096 && outer * inner >= 65536) ||
                 (red_n <= (outer * inner >= 131072 ? 16 : 12) && red_n * outer * inner < (13 << 16) * (int64_t)kvec);
  p.vec = inner >= kvec;
  const int64_t groups = p.vec ? cdiv(inner, kvec) : inner;
  // 16 column groups (256 bytes of a row) per block; fewer for narrower rows, so that the block's
  // other threads take more rows side by side
  p.cg_log2 = 4;
  if (!p.vec) p.cg_log2 = 3;
  while (p.cg_log2 > 0 && (1 << (p.cg_log2 - 1)) >= groups) --p.cg_log2;
  // More, up to 64, while that leaves 2048 blocks: every thread then has rows of its own to add where few
  // rows leave row groups idle, and fewer sums to combine where there are many. Past 64 only for fewer rows
  // than row groups. (us, one thread per output / 16 / as chosen: f16 sum over dim 0 of [5, 4000000] 17.7 /
  // 31 / 12.1, [64, 4000000] 240 / 94 / 90, fp32 over dim 1 of [64, 8, 65536] 42 / 54 / 26, [1000, 2, 4096]
  // 11.6 / 46 / 9.1; with 1024 blocks f16 [256, 262144] 22 / 26.)
  if (p.vec && p.cg_log2 == 4)
    while (p.cg_log2 < 8 && (p.cg_log2 < 6 || (kColThreads >> p.cg_log2) > red_n) &&
           cdiv(groups, (int64_t)2 << p.cg_log2) * outer >= 2048)
      ++p.cg_log2;
  p.col_blocks = cdiv(groups, (int64_t)1 << p.cg_log2);
  const int64_t rg = kColThreads >> p.cg_log2;
  const int64_t blocks = p.col_blocks * outer;
  const int64_t per_thread = cdiv(red_n, rg);
  // Slices: only where a thread would walk more than 32 rows (four rounds of loads, about what the
  // second launch costs) and the grid leaves the chip short of blocks; each slice keeps at least one
  // full round of loads per thread.
  p.slices = 1;
  if (blocks < 512 && per_thread > 32) p.slices = std::min<int64_t>(cdiv(1024, blocks), per_thread / kColUnroll);
  p.slice_rows = cdiv(cdiv(red_n, p.slices), rg) * rg;
  p.slices = red_n > 0 ? cdiv(red_n, p.slice_rows) : 1;
  return p;
}

template <typename T, typename TO, bool MAX>
static void launch_cols(const ColPlan& p, const typename T::S* x, typename TO::S* y, float* part, int64_t outer,
                        int64_t red_n, int64_t inner, hipStream_t s) {
  const dim3 grid((unsigned)(p.col_blocks * outer), (unsigned)p.slices);
  if (p.vec)
    reduce_cols<T, TO, T::kVec, MAX><<<grid, kColThreads, 0, s>>>(x, y, part, red_n, inner, p.cg_log2,
                                                                  (int)p.col_blocks, p.slice_rows);
  else
    reduce_cols<T, TO, 1, MAX><<<grid, kColThreads, 0, s>>>(x, y, part, red_n, inner, p.cg_log2,
                                                            (int)p.col_blocks, p.slice_rows);
}

template <typename T, bool MAX>
static int launch_reduce(const void* x, void* y, int64_t outer, int64_t red_n, int64_t inner,
                         float* ws, int64_t ws_bytes, hipStream_t s) {
  using S = typename T::S;
  const S* xp = (const S*)x;
  S* yp = (S*)y;
  if (inner == 1) {
    const int64_t rows = outer, cols = red_n;
    RowPlan plan;
    const bool any = cols % T::kVec != 0 || !host_aligned16(x);
    bool handled = false;
    if (plan_row_cols(rows, cols, T::kVec, any, &plan, 2)) {
      AK_ANY_SWITCH(any, AK_ROW_SWITCH({
        const dim3 grid((unsigned)cdiv(rows, RowGeom<L>::kRowsPerBlock));
        reduce_rows<T, L, VPT, MAX, ANY><<<grid, RowGeom<L>::kThreads, 0, s>>>(xp, yp, rows, (int)cols);
      }));
    }
    if (!handled) reduce_loop<T, MAX><<<(unsigned)rows, kLoopThreads, 0, s>>>(xp, yp, (int)cols);
    return record_launch();
  }
  ColPlan p = plan_cols(outer, red_n, inner, T::kVec);
  // (a block of the column kernel takes two to four threads per output, or more where inner is narrow, so
  // one thread per output still fits where its grid does not)
  if (p.short_rows || !grid_fits(p.col_blocks * outer, kColThreads)) {
    reduce_cols_short<T, MAX><<<(unsigned)cdiv(outer * inner, 256), 256, 0, s>>>(xp, yp, outer, red_n, inner);
    return record_launch();
  }
  if (p.slices > 1 && (!ws || ws_bytes < p.slices * outer * inner * (int64_t)sizeof(float))) {
    p.slices = 1;
    p.slice_rows = red_n;
  }
  if (p.slices == 1) {
    launch_cols<T, T, MAX>(p, xp, yp, nullptr, outer, red_n, inner, s);
    return record_launch();
  }
  launch_cols<T, T, MAX>(p, xp, yp, ws, outer, red_n, inner, s);
  // the slices of every output: [slices][outer * inner] reduced over its first dim
  ColPlan q = plan_cols(1, p.slices, outer * inner, TF32::kVec);
  q.slices = 1;
  q.slice_rows = p.slices;
  launch_cols<TF32, T, MAX>(q, ws, yp, nullptr, 1, p.slices, outer * inner, s);
  return record_launch();
}

}  // namespace ak

using namespace ak;

static bool bad_rows(int64_t rows, int64_t cols) {
  return rows < 0 || cols < 0 || cols > INT_MAX || rows > (int64_t)INT_MAX;
}

extern "C" int ak_rmsnorm(int dtype, const void* x, const void* w, void* y, int64_t rows,
                          int64_t cols, float eps, hipStream_t stream) {
  if (bad_rows(rows, cols)) return AK_EINVAL;
  if (rows == 0 || cols == 0) return AK_OK;
  if (!x || !w || !y) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_rmsnorm<T, 0>(x, w, y, rows, cols, eps, stream));
}

extern "C" int ak_rmsnorm_rsqrt(int dtype, const void* x, const void* w, void* y, int64_t rows,
                                int64_t cols, float eps, hipStream_t stream) {
  if (bad_rows(rows, cols)) return AK_EINVAL;
  if (rows == 0 || cols == 0) return AK_OK;
  if (!x || !w || !y) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_rmsnorm<T, 1>(x, w, y, rows, cols, eps, stream));
}

extern "C" int ak_layernorm(int dtype, const void* x, const void* w, const void* b, void* y,
                            int64_t rows, int64_t cols, float eps, hipStream_t stream) {
  if (bad_rows(rows, cols)) return AK_EINVAL;
  if (rows == 0 || cols == 0) return AK_OK;
  if (!x || !y) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_layernorm<T>(x, w, b, y, rows, cols, eps, stream));
}

extern "C" int ak_softmax(int dtype, const void* x, void* y, int64_t rows, int64_t cols,
                          hipStream_t stream) {
  // a call that launches nothing still consumes pending launch events (they never carry over)
  const bool launches = !bad_rows(rows, cols) && rows != 0 && cols != 0 && x && y &&
                        (dtype == AK_F32 || dtype == AK_F16 || dtype == AK_BF16);
  if (!launches) take_launch_events();
  if (bad_rows(rows, cols)) return AK_EINVAL;
  if (rows == 0 || cols == 0) return AK_OK;
  if (!x || !y) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_softmax<T>(x, y, rows, cols, stream));
}

extern "C" int ak_cross_entropy(int dtype, const void* logits, const int64_t* targets,
                                float* row_loss, void* out, int64_t rows, int64_t vocab,
                                int64_t ignore_index, hipStream_t stream) {
  if (bad_rows(rows, vocab)) return AK_EINVAL;
  if (!out) return AK_EINVAL;
  if (rows > 0 && (!logits || !targets || !row_loss || vocab == 0)) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_ce<T>(logits, targets, row_loss, out, rows, vocab, ignore_index, stream));
}

// ---------------------------------------------------------------------------------------------
// ak_cross_entropy_noalloc: ak_cross_entropy with the per-row losses in a file-scope device array
// instead of a caller workspace, for callers that cannot allocate. In host code `scratch` names a
// host-side stand-in, not device memory: its device address is looked up once per device with
// hipGetSymbolAddress (that device current) and cached; kernels only ever get that address.
// Every call writes the loss of each of its rows before ce_mean reads it, so nothing has to be
// cleared between calls; calls that overlap on one device share the array and race.
// ---------------------------------------------------------------------------------------------
static __device__ __align__(256) float scratch[AK_CE_NOALLOC_MAX_ROWS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
std::atomic<float*> g_scratch[kMaxDevices];

// Device address of `scratch` on the device that runs `stream` (the current device for the null
// stream); AK_OK or an error status.
int ce_scratch(hipStream_t stream, float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess && stream) e = hipStreamGetDevice(stream, &dev);
  if (e != hipSuccess) return record_hip_error(e);
  if (dev < 0 || dev >= kMaxDevices) return AK_EUNSUPPORTED;
  float* p = g_scratch[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch[dev].load(std::memory_order_relaxed);
    if (!p) {
      int cur = dev;
      e = hipGetDevice(&cur);
      if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
      void* addr = nullptr;
      if (e == hipSuccess) e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
      if (cur != dev) {
        const hipError_t e2 = hipSetDevice(cur);
        if (e == hipSuccess) e = e2;
      }
      if (e != hipSuccess) return record_hip_error(e);
      if (!addr) return AK_EHIP;
      p = static_cast<float*>(addr);
      g_scratch[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return AK_OK;
}
}  // namespace

extern "C" int ak_cross_entropy_noalloc(int dtype, const void* logits, const int64_t* targets, void* out,
                                        int64_t rows, int64_t vocab, int64_t ignore_index, hipStream_t stream) {
  if (bad_rows(rows, vocab)) return AK_EINVAL;
  if (rows > AK_CE_NOALLOC_MAX_ROWS) return AK_EINVAL;
  if (!out) return AK_EINVAL;
  if (rows > 0 && (!logits || !targets || vocab == 0)) return AK_EINVAL;
  if (dtype != AK_F32 && dtype != AK_F16 && dtype != AK_BF16) return AK_EINVAL;
  float* loss = nullptr;
  const int st = ce_scratch(stream, &loss);
  if (st != AK_OK) return st;
  AK_DISPATCH(dtype, T, return launch_ce<T>(logits, targets, loss, out, rows, vocab, ignore_index, stream));
}

static bool bad_reduce(int64_t outer, int64_t reduce, int64_t inner) {
  return outer < 0 || reduce < 0 || inner < 0 || reduce > INT_MAX || outer > (int64_t)INT_MAX * 256;
}

extern "C" int64_t ak_reduce_workspace_bytes(int dtype, int64_t outer, int64_t reduce, int64_t inner) {
  if (dtype != AK_F32 && dtype != AK_F16 && dtype != AK_BF16) return 0;
  if (bad_reduce(outer, reduce, inner) || outer == 0 || inner <= 1 || reduce == 0) return 0;
  const ColPlan p = plan_cols(outer, reduce, inner, dtype == AK_F32 ? TF32::kVec : TF16::kVec);
  if (p.short_rows || p.slices <= 1) return 0;
  return p.slices * outer * inner * (int64_t)sizeof(float);
}

extern "C" int ak_reduce_sum_ws(int dtype, const void* x, void* y, int64_t outer, int64_t reduce, int64_t inner,
                                void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (bad_reduce(outer, reduce, inner)) return AK_EINVAL;
  if (outer == 0 || inner == 0) return AK_OK;
  if (!x || !y || (((uintptr_t)workspace) & 3u)) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_reduce<T, false>(x, y, outer, reduce, inner, (float*)workspace,
                                                       workspace_bytes, stream));
}

extern "C" int ak_reduce_max_ws(int dtype, const void* x, void* y, int64_t outer, int64_t reduce, int64_t inner,
                                void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (bad_reduce(outer, reduce, inner) || reduce == 0) return AK_EINVAL;
  if (outer == 0 || inner == 0) return AK_OK;
  if (!x || !y || (((uintptr_t)workspace) & 3u)) return AK_EINVAL;
  AK_DISPATCH(dtype, T, return launch_reduce<T, true>(x, y, outer, reduce, inner, (float*)workspace,
                                                      workspace_bytes, stream));
}

extern "C" int ak_reduce_sum(int dtype, const void* x, void* y, int64_t outer, int64_t reduce,
                             int64_t inner, hipStream_t stream) {
  return ak_reduce_sum_ws(dtype, x, y, outer, reduce, inner, nullptr, 0, stream);
}

extern "C" int ak_reduce_max(int dtype, const void* x, void* y, int64_t outer, int64_t reduce,
                             int64_t inner, hipStream_t stream) {
  return ak_reduce_max_ws(dtype, x, y, outer, reduce, inner, nullptr, 0, stream);
}

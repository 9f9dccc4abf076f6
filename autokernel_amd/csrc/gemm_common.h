// gemm_common.h -- what the GEMM sources share: tile order, epilogue arguments and
// the epilogue applied to a lane's accumulators (gemm.hip, gemm_f32.hip).
#pragma once
#include "mfma.h"

namespace ak {

// 4x8 transpose of 16-bit values: in[r] holds 8 n-values of k-row r; out[n] gets the 4 k-values
// of column n (v_perm_b32 picks the low or high halves of two words).
__device__ __forceinline__ void transpose4x8(const u32x4 (&in)[4], u32x2 (&out)[8]) {
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int w = n >> 1;
    const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
    out[n][0] = __builtin_amdgcn_perm(in[1][w], in[0][w], sel);
    out[n][1] = __builtin_amdgcn_perm(in[3][w], in[2][w], sel);
  }
}

// Tile scheduling: logical tile index for this block (XCD-aware, grouped along M).
__device__ __forceinline__ void tile_coords(int tiles_m, int tiles_n, int* tm, int* tn) {
  const int nb = gridDim.x;
  const int bid = blockIdx.x;
  const int full = nb & ~7;
  const int L = bid < full ? (bid & 7) * (full >> 3) + (bid >> 3) : bid;
  constexpr int GM = 4;
  const int per_group = GM * tiles_n;
  const int g = L / per_group;
  const int first_m = g * GM;
  const int gsz = min(tiles_m - first_m, GM);
  const int r = L - g * per_group;
  *tm = first_m + r % gsz;
  *tn = r / gsz;
}

// --------------------------------------------------------------------------------------------
// Epilogues (applied to fp32 accumulators; every step rounds like the reference's tensor ops)
// --------------------------------------------------------------------------------------------
enum Epi { kEpiStore = 0, kEpiSilu = 1, kEpiGelu = 2, kEpiRelu2 = 3, kEpiNone = 4, kEpiResidual = 5, kEpiRope = 6,
           kEpiPartial = 7, kEpiBias = 8, kEpiBiasGelu = 9, kEpiBiasResidual = 10 };

// Arguments of the rotary epilogue (kEpiRope), passed by value to every f16 / bf16 GEMM kernel:
// columns [0, rot_cols) of C form heads of head_dim columns whose (even, odd) pairs are rotated
// by the fp32 tables cos / sin [seq_len, head_dim / 2]; row m of C is token m % seq_len.
//
// Split-K (kEpiPartial): the grid's y dimension is the K slice; slice z multiplies A and B advanced
// by z * split_a / z * split_b elements and stores its fp32 accumulators to the workspace advanced by
// z * split_c floats (row stride ldc), for splitk_reduce to sum.
struct EpiArgs {
  const uint16_t* bias = nullptr;  // kEpiBiasResidual (R is the residual there)
  const float* cos = nullptr;
  const float* sin = nullptr;
  int head_dim = 0;
  int rot_cols = 0;
  int seq_len = 1;
  int splits = 1;
  int64_t split_a = 0, split_b = 0, split_c = 0;
  // Batched products (ak_gemm_batched): grid z is the batch item; item z reads A and B advanced by
  // z * batch_a / z * batch_b elements and writes C advanced by z * batch_c (a stride of 0 shares
  // the operand across the batch).
  int batch = 1;
  int64_t batch_a = 0, batch_b = 0, batch_c = 0;
  // Items skip, skip + skip_period, ... are another launch's (their operands are 16-byte aligned, the others'
  // are not); -1: none.
  int skip = -1, skip_period = 1;
};

__device__ __forceinline__ bool skip_item(const EpiArgs& ep) {
  return ep.skip >= 0 && (int)blockIdx.z % ep.skip_period == ep.skip;
}

// Bases of this block's batch item (grid z); one item when ep.batch == 1.
template <class PA, class PB, class PC>
__device__ __forceinline__ void batch_bases(PA& A, PB& B, PC& C, const EpiArgs& ep) {
  if (ep.batch > 1) {
    const int64_t z = blockIdx.z;
    A += z * ep.batch_a;
    B += z * ep.batch_b;
    C += z * ep.batch_c;
  }
}

// The model's rotation of one pair in fp32, each product and sum rounded on its own (no fused
// multiply-add), as separate fp32 tensor ops compute (a c - b s, a s + b c).
__device__ __forceinline__ void rope_rotate(float& a, float& b, float c, float s) {
#pragma clang fp contract(off)
  const float y1 = a * c - b * s;
  const float y2 = a * s + b * c;
  a = y1;
  b = y2;
}

// torch's exact GELU of one rounded value, in fp32: x * 0.5 * (1 + erf(x / sqrt(2)))
__device__ __forceinline__ float gelu_erf(float g) { return 0.5f * g * (1.0f + erff(g * 0.70710678118654752f)); }

template <typename T, int EPI>
__device__ __forceinline__ float gate_up(float g_acc, float u_acc) {
  const float g = T::rnd(g_acc);
  const float u = T::rnd(u_acc);
  float a;
  if constexpr (EPI == kEpiSilu) a = T::rnd(g / (1.0f + expf(-g)));
  else if constexpr (EPI == kEpiGelu) a = T::rnd(gelu_erf(g));
  else if constexpr (EPI == kEpiRelu2) { const float r = g > 0.f ? g : 0.f; a = T::rnd(r * r); }
  else a = g;
  return a * u;  // rounded by the store
}

// Epilogue of one lane's share of a block tile: for fragment (i, j) the lane holds the four
// consecutive outputs C[m][n .. n + 3], m = mb + MST i, n = nb + NST j, in acc[.][i][j] (NB == 2:
// gate and up accumulators, combined by gate_up).
//   kEpiResidual rounds the product to the element type, adds R[m][n + e] (R shares C's leading
//     dimension) and rounds again: the two roundings of torch's `R + A @ B`. fp32 holds the sum of
//     two f16 / bf16 values to 24 bits, at least 2p + 2 for both formats, so rounding it once more
//     gives the correctly rounded sum.
//   kEpiBias adds bias[n + e] (the element type, R points at it) to the fp32 accumulator and
//     rounds once: nn.Linear's fused bias (torch's addmm adds it in the fp32 compute type).
//   kEpiBiasGelu is kEpiBias's rounded value through exact GELU in fp32, rounded again: a biased
//     nn.Linear followed by nn.GELU (R points at the bias).
//   kEpiBiasResidual is kEpiBias's rounded value plus R[m][n + e] (the residual; the bias comes
//     from ep.bias), rounded again: torch's `R + linear(x)` for a biased Linear.
//   kEpiRope rounds the product to the element type, then (columns below rot_cols) rotates the
//     pairs (n, n + 1), (n + 2, n + 3) in fp32 by table row m % seq_len and rounds once: the
//     projection's output cast to fp32, rotated and cast back. n is a multiple of 4 and head_dim
//     of 4, so the four columns never straddle a head or the rot_cols boundary.
// The side values (R, or the cos / sin pairs) of every fragment are loaded first, then combined
// and stored, so their latency is paid once per tile rather than once per fragment.
// Stores: the results of fragments 2p and 2p + 1 (columns 32p + 4g + 0..3 and 32p + 16 + 4g + 0..3
// in lane group g = lane / 16) are packed to the element type and regrouped across the four lane
// groups (regroup8), so each lane stores 8 consecutive columns 32p + 8g + 0..7 of its row: one
// 16-byte store where C is 16-byte aligned, which fills the 64-byte requests (4 lanes x 16 bytes
// per row) that 8-byte stores half-fill.
// VEC: a lane's 8 in-range columns of C are one 16-byte store at any alignment (store_cols), so
// any leading dimension works (an odd ldc, e.g. a 50257-column vocabulary projection); R's four
// columns load as one 8-byte access where that is 8-byte aligned, as elements otherwise.
// Regroup two fragments' packed columns across the 16-lane groups of a wave. On entry lane group g
// (lanes 16g .. 16g + 15) holds 4-column group g of fragment x and of fragment y, i.e. groups g and
// 4 + g of their 32 columns; on exit it holds group 2g in x and group 2g + 1 in y. Lanes keep their
// row (lane % 16). permlane32_swap exchanges x's upper half-wave with y's lower one
// (x = [x0 x1 y0 y1], y = [x2 x3 y2 y3] by lane group), permlane16_swap x's odd lane groups with
// y's even ones (x = [x0 x2 y0 y2], y = [x1 x3 y1 y3]).
__device__ __forceinline__ void regroup8(uint32_t& x, uint32_t& y) {
  const auto h = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  const auto q = __builtin_amdgcn_permlane16_swap(h[0], h[1], false, false);
  x = q[0];
  y = q[1];
}

// Store the first W (4 or 8) 16-bit elements of o (element e in dword e / 2, low half first) to
// cp[0 .. W - 1], the first `valid` of them only. With all W in range (VEC) it is one 16- or 8-byte
// store at whatever 2-byte alignment cp has: global memory on this target takes multi-dword
// accesses at any alignment (the HSA code object is built with unaligned-access-mode, which is why
// the compiler emits one global_store_dwordx4 for a 2-byte-aligned pointer here). Rows whose start
// is not 16-byte aligned (an odd ldc, e.g. a 50257-column vocabulary projection) took 47 % longer
// with stores narrowed to their alignment.
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
template <bool VEC, int W>
__device__ __forceinline__ void store_cols(uint16_t* cp, int valid, const u32x4& o) {
  if (VEC && valid >= W) {
    if constexpr (W == 8) *reinterpret_cast<u32x4_a2*>(cp) = o;
    else *reinterpret_cast<u32x2_a2*>(cp) = u32x2{o[0], o[1]};
    return;
  }
#pragma unroll
  for (int e = 0; e < W; ++e)
    if (e < valid) cp[e] = (uint16_t)(o[e >> 1] >> ((e & 1) * 16));
}

template <typename T, int NB, int EPI, bool VEC, int FM, int FN, int MST = 16, int NST = 16>
__device__ __forceinline__ void tile_epilogue(uint16_t* __restrict__ C, const uint16_t* __restrict__ R,
                                              int64_t ldc, int M, int N, int mb, int nb,
                                              const f32x4 (&acc)[NB][FM][FN], const EpiArgs& ep) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  constexpr bool kRes = NB == 1 && (EPI == kEpiResidual || EPI == kEpiBiasResidual);
  constexpr bool kRope = NB == 1 && EPI == kEpiRope;
  constexpr bool kBias = NB == 1 && (EPI == kEpiBias || EPI == kEpiBiasGelu || EPI == kEpiBiasResidual);
  if constexpr (NB == 1 && EPI == kEpiPartial) {
    // fp32 accumulators as they are (C is the fp32 workspace; N % 4 == 0 and ldc % 4 == 0)
    float* Cf = reinterpret_cast<float*>(C);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = mb + i * MST;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = nb + j * NST;
        if (n < N) *reinterpret_cast<f32x4*>(Cf + (int64_t)m * ldc + n) = acc[0][i][j];
      }
    }
    return;
  }
  u32x2 side_r[kRes ? FM : 1][kRes ? FN : 1];
  float side_b[kBias ? FN : 1][4];
  if constexpr (kBias) {
    const uint16_t* bias = EPI == kEpiBiasResidual ? ep.bias : R;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = nb + j * NST;
#pragma unroll
      for (int e = 0; e < 4; ++e) side_b[j][e] = n + e < N ? T::to_f(bias[n + e]) : 0.f;
    }
  }
  f32x2 side_c[kRope ? FM : 1][kRope ? FN : 1], side_s[kRope ? FM : 1][kRope ? FN : 1];
  if constexpr (kRes) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int m = mb + i * MST, n = nb + j * NST;
        const uint16_t* rp = R + (int64_t)m * ldc + n;
        u32x2 r = {0u, 0u};
        if (m < M) {
          if (VEC && n + 3 < N && ((uintptr_t)rp & 7u) == 0) {
            r = *reinterpret_cast<const u32x2*>(rp);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < N) r[e >> 1] |= (uint32_t)rp[e] << ((e & 1) * 16);
          }
        }
        side_r[i][j] = r;
      }
  }
  if constexpr (kRope) {
    const int half = ep.head_dim >> 1;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = mb + i * MST;
      const int64_t row = (int64_t)((m < M ? m : 0) % ep.seq_len) * half;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = nb + j * NST;
        f32x2 c = {1.f, 1.f}, sn = {0.f, 0.f};
        if (n < ep.rot_cols) {
          const int64_t t = row + ((n % ep.head_dim) >> 1);  // even: 8-byte aligned pairs
          c = *reinterpret_cast<const f32x2*>(ep.cos + t);
          sn = *reinterpret_cast<const f32x2*>(ep.sin + t);
        }
        side_c[i][j] = c;
        side_s[i][j] = sn;
      }
    }
  }
  static_assert(NST == 16, "fragment pairs regroup 16-column fragments");
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = mb + i * MST;
    uint32_t lo[FN], hi[FN];  // packed columns 0, 1 and 2, 3 of each fragment
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = nb + j * NST;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (NB == 2) v[e] = gate_up<T, EPI>(acc[0][i][j][e], acc[1][i][j][e]);
        else if constexpr ((kRes && !kBias) || kRope) v[e] = T::rnd(acc[0][i][j][e]);
        else v[e] = acc[0][i][j][e];
      }
      if constexpr (kBias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] += side_b[j][e];
          if constexpr (EPI != kEpiBias) v[e] = T::rnd(v[e]);
          if constexpr (EPI == kEpiBiasGelu) v[e] = gelu_erf(v[e]);
        }
      }
      if constexpr (kRes) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += T::to_f((uint16_t)(side_r[i][j][e >> 1] >> ((e & 1) * 16)));
      }
      if constexpr (kRope) {
        if (n < ep.rot_cols) {
          rope_rotate(v[0], v[1], side_c[i][j][0], side_s[i][j][0]);
          rope_rotate(v[2], v[3], side_c[i][j][1], side_s[i][j][1]);
        }
      }
      lo[j] = (uint32_t)T::from_f(v[0]) | ((uint32_t)T::from_f(v[1]) << 16);
      hi[j] = (uint32_t)T::from_f(v[2]) | ((uint32_t)T::from_f(v[3]) << 16);
    }
    // fragment pairs: 8 consecutive columns per lane (the shuffles run on every lane, before the
    // row test)
    const int g = (lane_id() >> 4) & 3;
    const int nq = nb - 4 * g + 8 * g;  // lane group g's first column of pair 0
#pragma unroll
    for (int j = 0; j + 1 < FN; j += 2) {
      regroup8(lo[j], lo[j + 1]);
      regroup8(hi[j], hi[j + 1]);
      if (m < M) {
        const u32x4 o = {lo[j], hi[j], lo[j + 1], hi[j + 1]};
        const int n = nq + j * NST;
        store_cols<VEC, 8>(C + (int64_t)m * ldc + n, N - n, o);
      }
    }
    if constexpr (FN % 2 == 1) {
      if (m < M) {
        const int n = nb + (FN - 1) * NST;
        const u32x4 o = {lo[FN - 1], hi[FN - 1], 0u, 0u};
        store_cols<VEC, 4>(C + (int64_t)m * ldc + n, N - n, o);
      }
    }
  }
}

// Products with at most kSmallM rows of A (gemm_small.hip); any alignment, any K > 0. N stays below the
// 2^32 work-items of a grid: at most 16 per column (32 for gate/up).
constexpr int64_t kSmallM = 64;
constexpr int64_t small_max_n(int nb) { return ((int64_t)1 << 28) / nb - 64; }
// gemm_small for one product of N <= 4096 columns: whether its waves take groups of two k-steps (of one
// else), and its blocks.
inline bool small_k64(int64_t M, int64_t N, bool bt) { return M <= 16 || N <= 1024 || (bt && M <= 32); }
inline int64_t small_blocks(int64_t M, int64_t N, bool bt) {
  const bool one = M <= 16 || N <= 1024;  // 16 rows a block
  return cdiv(M, one ? 16 : 32) * cdiv(N, bt && (one || M <= 32) ? 16 : 32);
}
template <typename T, int NB, int EPI>
int launch_gemm_small(const void* A, const void* B0, const void* B1, void* C, int64_t M, int64_t N, int64_t K,
                      int64_t lda, int64_t ldb, int64_t ldc, bool bt, hipStream_t s, const EpiArgs& ep);

// fp32 products (gemm_f32.hip). batch > 1: grid z is the batch item, whose operands start z * batch_x
// elements further.
int launch_gemm32(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda,
                  int64_t ldb, int64_t ldc, bool bt, hipStream_t s, int batch = 1, int64_t batch_a = 0,
                  int64_t batch_b = 0, int64_t batch_c = 0);
// fp32 gate/up: H = act(x Wg^T) * (x Wu^T); epi is an Epi activation.
int launch_gate_up32(const void* x, const void* wg, const void* wu, void* h, int64_t M, int64_t H, int64_t D,
                     int epi, hipStream_t s);

}  // namespace ak

// attention_rows.hip -- flash-attention forward for few query rows per KV head (decode: one new query
// per sequence against its cached keys), f16 / bf16, head_dim 64 or 128.
//
// What bounds it: reading K and V once from HBM. fa_fwd2 gives every query head a block of 128 query
// rows, so a decode step reads each KV head `group` times for one useful row per block and walks the
// keys serially in few blocks. Here the group x Sq query rows of a KV head (16 per block) are the
// columns of one MFMA tile, and the keys are split over the waves of a block and over `splits` blocks:
//   * A wave takes 32 keys per step, straight from global memory into registers (no LDS, no
//     barrier), the next step's loads in flight while it computes.
//   * S^T = K Q^T on v_mfma_f32_16x16x32: two 16-key tiles whose row i of tile t is key
//     8 (i / 4) + 4 t + i % 4, so the lanes of group g = lane / 16 end up with the scores of keys
//     8 g .. 8 g + 7 of one query: in order, the B operand of the next product.
//   * O^T += V^T P^T: a lane loads D / 16 consecutive dims of eight keys (one row of V per 16 lanes,
//     whole cache lines) and transposes them in registers (v_perm_b32) into the A operands of D / 16
//     fragments, fragment e holding dims (D / 16) i + e.
//   * Online softmax per wave (exact running max, P <= 1 rounded to the element type, row sums of the
//     rounded weights, as fa_fwd2), merged over the block's waves through LDS and, with splits > 1,
//     over blocks by fa_rows_merge from fp32 partials in the caller's workspace, in a fixed order.
// Measured, bf16: [8, 32/8, 1 x 4096, 128] 82.9 -> 30.1 us, [1, 4, 1 x 17914, 128] 199 -> 19.7 us,
// [1, 32, 1 x 32768, 128] 366 -> 95 us (5.6 TB/s).
#include <limits.h>

#include <algorithm>

#include "attention_common.h"
#include "mfma.h"

namespace ak {

constexpr int kFrWaves = 4;
constexpr int kFrThreads = kFrWaves * kWave;
constexpr int kFrRows = 16;  // query rows per block (MFMA columns)
constexpr int kFrKeys = 32;  // keys per wave and step
constexpr int kFrMaxSplits = 64;

struct FrArgs {
  const uint16_t *Q, *K, *V;
  uint16_t* O;
  float *part, *stat;  // [splits][total rows][D] and [splits][total rows][4] (base, sum, true max)
  int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss, osb, osh, oss;
  int Hkv, group, Sq, Sk, rows, row_blocks, splits, split_keys;
  int64_t total;  // B * Hq * Sq
  float c_log2, thr;
};

// max / sum over the four 16-lane groups of a wave (every lane gets the result)
struct OpMaximum {
  __device__ __forceinline__ float operator()(float a, float b) const { return fa2_max(a, b); }
};
template <typename Op>
__device__ __forceinline__ float fr_groups(float v, Op op) {
  return wave_step<5>(wave_step<4>(v, op), op);
}

template <int D>
struct FrVec;  // D / 16 16-bit values of one V row
template <>
struct FrVec<128> {
  typedef u32x4 type;
};
template <>
struct FrVec<64> {
  typedef u32x2 type;
};

template <typename T, int D>
__device__ __forceinline__ void fr_store_row(const FrArgs& a, int64_t row, int c, const float (&o)[D / 16], float l,
                                             float mt) {
  constexpr int VW = D / 16;
  // row = (bh * rows + r), r = head in group * Sq + query
  const int64_t bh = row / a.rows;
  const int r = (int)(row - bh * a.rows);
  const int b = (int)(bh / a.Hkv), h = (int)(bh - (int64_t)b * a.Hkv) * a.group + r / a.Sq;
  const bool nan_row = !(mt < a.thr && mt > -a.thr);  // as fa_fwd2
  const float inv = nan_row ? __builtin_nanf("") : 1.0f / l;
  typename FrVec<D>::type pk;
#pragma unroll
  for (int e = 0; e < VW / 2; ++e) pk[e] = fa2_pack<T>(o[2 * e] * inv, o[2 * e + 1] * inv);
  *reinterpret_cast<typename FrVec<D>::type*>(a.O + b * a.osb + h * a.osh + (r % a.Sq) * a.oss + c * VW) = pk;
}

template <typename T, int D>
__global__ __launch_bounds__(kFrThreads, 2) void fa_rows(const FrArgs a) {
  constexpr int NS = D / 32;  // 32-deep steps of S^T
  constexpr int VW = D / 16;  // V elements per lane and key; O^T fragments
  using VV = typename FrVec<D>::type;
  __shared__ __attribute__((aligned(16))) float so[kFrWaves][kFrRows][D + 4];
  __shared__ float sst[kFrWaves][kFrRows][3];

  const int sp = (int)(blockIdx.x % (unsigned)a.splits);
  const int rest = (int)(blockIdx.x / (unsigned)a.splits);
  const int rb = rest % a.row_blocks;
  const int64_t bh = rest / a.row_blocks;
  const int b = (int)(bh / a.Hkv), hk = (int)(bh % a.Hkv);
  const int lane = lane_id(), w = wave_id();
  const int i16 = lane & 15, g = lane >> 4;
  const uint16_t* Kb = a.K + b * a.ksb + hk * a.ksh;
  const uint16_t* Vb = a.V + b * a.vsb + hk * a.vsh;

  // Q: the B operand, column i16 = query row rb * 16 + i16 of this KV head
  const int r = rb * kFrRows + i16;
  u32x4 qf[NS];
  {
    const uint16_t* q = a.Q + b * a.qsb + (int64_t)(hk * a.group + r / a.Sq) * a.qsh + (int64_t)(r % a.Sq) * a.qss;
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = r < a.rows ? ld16(q + s * 32 + g * 8) : u32x4{0u, 0u, 0u, 0u};
  }

  const int kbeg = sp * a.split_keys, kend = min(a.Sk, kbeg + a.split_keys);
  struct Step {
    u32x4 k[2][NS];
    VV v[8];
  };
  // Keys past the slice's end read its last key (K; their scores are masked) or come as zeros (V).
  auto load = [&](int k0, Step& st) {
    const bool tail = k0 + kFrKeys > kend;  // uniform
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      int key = k0 + 8 * (i16 >> 2) + 4 * t + (i16 & 3);
      if (tail) key = min(key, kend - 1);
      const uint16_t* p = Kb + (int64_t)key * a.kss + g * 8;
#pragma unroll
      for (int s = 0; s < NS; ++s) st.k[t][s] = ld16(p + s * 32);
    }
    const uint16_t* p = Vb + (int64_t)(k0 + 8 * g) * a.vss + i16 * VW;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (!tail || k0 + 8 * g + e < kend) {
        st.v[e] = *reinterpret_cast<const VV*>(p + (int64_t)e * a.vss);
      } else {
#pragma unroll
        for (int x = 0; x < VW / 2; ++x) st.v[e][x] = 0u;
      }
    }
  };

  f32x4 o[VW];
#pragma unroll
  for (int e = 0; e < VW; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, m_true = -INFINITY, l_run = 0.f;  // l_run: this lane's keys only
  auto compute = [&](int k0, const Step& st) {
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
      for (int t = 0; t < 2; ++t) s[t] = mfma16x16x32<T>(st.k[t][x], qf[x], s[t]);
    if constexpr (T::kCode == AK_F16) {
      // f16 scores round to -inf past the range and weigh nothing, however small the scale. (One at the
      // other end makes its row NaN, see fr_store_row.)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (s[t][v] <= -a.thr) s[t][v] = -INFINITY;
    }
    if (k0 + kFrKeys > kend) {
      const int left = kend - (k0 + 8 * g);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (4 * t + v >= left) s[t][v] = -INFINITY;
    }
    float mt = fa2_max(fa2_max(s[0][0], s[0][1]), fa2_max(s[0][2], s[0][3]));
    mt = fa2_max(mt, fa2_max(fa2_max(s[1][0], s[1][1]), fa2_max(s[1][2], s[1][3])));
    mt = fr_groups(mt, OpMaximum());
    m_true = fa2_max(m_true, mt);
    const float m_new = fmaxf(m_run, mt * a.c_log2);
    const float base = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = m_new == m_run ? 1.0f : __builtin_amdgcn_exp2f(m_run - base);
    m_run = m_new;
    u32x4 pf;
    float ps = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e >> 1][2 * (e & 1)], a.c_log2, -base));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e >> 1][2 * (e & 1) + 1], a.c_log2, -base));
      pf[e] = fa2_pack<T>(p0, p1);
      ps = fa2_sum2<T>(pf[e], ps);
    }
    l_run = l_run * alpha + ps;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int e = 0; e < VW; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v) o[e][v] *= alpha;
    }
#pragma unroll
    for (int e = 0; e < VW; ++e) {
      const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
      u32x4 vt;
#pragma unroll
      for (int p = 0; p < 4; ++p) vt[p] = __builtin_amdgcn_perm(st.v[2 * p + 1][e >> 1], st.v[2 * p][e >> 1], sel);
      o[e] = mfma16x16x32<T>(vt, pf, o[e]);
    }
  };

  constexpr int kStride = kFrWaves * kFrKeys;
  int k0 = kbeg + w * kFrKeys;
  if (k0 < kend) {
    Step s0, s1;
    load(k0, s0);
    while (true) {
      const bool more1 = k0 + kStride < kend;
      if (more1) load(k0 + kStride, s1);
      compute(k0, s0);
      if (!more1) break;
      k0 += kStride;
      const bool more0 = k0 + kStride < kend;
      if (more0) load(k0 + kStride, s0);
      compute(k0, s1);
      if (!more0) break;
      k0 += kStride;
    }
  }
  l_run = fr_groups(l_run, OpAdd());

  // Merge the waves: lane (i16, g) holds of query i16, in o[e][v], dim VW (4 g + v) + e.
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int e = 0; e < VW; ++e) so[w][i16][VW * (4 * g + v) + e] = o[e][v];
  if (g == 0) {
    sst[w][i16][0] = m_run;
    sst[w][i16][1] = l_run;
    sst[w][i16][2] = m_true;
  }
  __syncthreads();
  const int q = threadIdx.x >> 4, c = threadIdx.x & 15;  // query row of the block, VW dims at c * VW
  if (rb * kFrRows + q >= a.rows) return;
  float mb = -INFINITY, mt = -INFINITY, l = 0.f, acc[VW];
#pragma unroll
  for (int x = 0; x < kFrWaves; ++x) {
    mb = fmaxf(mb, sst[x][q][0]);
    mt = fa2_max(mt, sst[x][q][2]);
  }
#pragma unroll
  for (int e = 0; e < VW; ++e) acc[e] = 0.f;
#pragma unroll
  for (int x = 0; x < kFrWaves; ++x) {
    const float f = sst[x][q][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sst[x][q][0] - mb);
    l += sst[x][q][1] * f;
#pragma unroll
    for (int e = 0; e < VW; ++e) acc[e] += so[x][q][c * VW + e] * f;
  }
  const int64_t row = bh * a.rows + rb * kFrRows + q;
  if (a.splits == 1) {
    fr_store_row<T, D>(a, row, c, acc, l, mt);
    return;
  }
  float* p = a.part + ((int64_t)sp * a.total + row) * D + c * VW;
#pragma unroll
  for (int e = 0; e < VW; e += 4) *reinterpret_cast<f32x4*>(p + e) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
  if (c == 0) *reinterpret_cast<f32x4*>(a.stat + ((int64_t)sp * a.total + row) * 4) = f32x4{mb, l, mt, 0.f};
}

// O of one row from its `splits` partials, one block per row: thread (x, c) adds splits x, x + 16, ...
// of dims c VW .. c VW + VW - 1, and the 16 sums of each dim combine in a fixed tree.
template <typename T, int D>
__global__ __launch_bounds__(kFrThreads) void fa_rows_merge(const FrArgs a) {
  constexpr int VW = D / 16;
  __shared__ float red[16][16 * VW + 1], rl[16];
  const int64_t row = blockIdx.x;
  const int x = threadIdx.x >> 4, c = threadIdx.x & 15;
  const float* st = a.stat + row * 4;
  const float* p = a.part + row * D + c * VW;
  const int64_t sstep = a.total * 4, pstep = a.total * D;
  f32x4 z[4], v[4][VW / 4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {  // at most 64 splits: every load issued before the first use
    const int s = min(x + 16 * u, a.splits - 1);
    z[u] = *reinterpret_cast<const f32x4*>(st + s * sstep);
#pragma unroll
    for (int e = 0; e < VW / 4; ++e) v[u][e] = *reinterpret_cast<const f32x4*>(p + s * pstep + 4 * e);
  }
  // every thread takes the row's base and true max over all splits
  float mb = -INFINITY, mt = -INFINITY;
  for (int s = c; s < a.splits; s += 16) {
    mb = fmaxf(mb, st[s * sstep]);
    mt = fa2_max(mt, st[s * sstep + 2]);
  }
  mb = seg_reduce<16>(mb, OpMax());
  mt = seg_reduce<16>(mt, OpMaximum());
  float l = 0.f, acc[VW];
#pragma unroll
  for (int e = 0; e < VW; ++e) acc[e] = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (x + 16 * u >= a.splits) continue;  // loaded the last split again: 0 times its infinities would be NaN
    const float f = z[u][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(z[u][0] - mb);
    l += z[u][1] * f;
#pragma unroll
    for (int e = 0; e < VW; ++e) acc[e] += v[u][e >> 2][e & 3] * f;
  }
#pragma unroll
  for (int e = 0; e < VW; ++e) red[x][e * 16 + c] = acc[e];
  if (c == 0) rl[x] = l;
  for (int h = 8; h > 0; h >>= 1) {
    __syncthreads();
    if (x < h) {
#pragma unroll
      for (int e = 0; e < VW; ++e) red[x][e * 16 + c] += red[x + h][e * 16 + c];
      if (c == 0) rl[x] += rl[x + h];
    }
  }
  __syncthreads();
  if (x != 0) return;
#pragma unroll
  for (int e = 0; e < VW; ++e) acc[e] = red[0][e * 16 + c];
  fr_store_row<T, D>(a, row, c, acc, rl[0], mt);
}

FaRowsPlan fa_rows_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D, bool causal) {
  FaRowsPlan p{false, 1, 0};
  const int64_t rows = Hq / Hkv * Sq;
  // A causal call's keys end at its last query (top-left mask), so few rows see few keys. Past 16 rows
  // K and V are read once per 16: still less than fa_fwd2's once per head when the rows are the group's.
  if (causal || (D != 64 && D != 128) || Sk > INT_MAX / 2) return p;
  if (rows > kFrRows && (Sq > 4 || rows > 4 * kFrRows)) return p;
  const int64_t blocks = B * Hkv * cdiv(rows, kFrRows);
  if (blocks > INT_MAX / kFrMaxSplits || B * Hq * Sq > INT_MAX) return p;
  p.ok = true;
  // One block per CU (four waves, 32 KB in flight each, already reach the HBM rate: 512 or 1024 blocks
  // measured the same kernel time and a longer merge); slices of at least 256 keys, and none below 1536
  // keys, where the second launch costs more than the shorter walk saves ([1, 8, 1 x 1024, 128]: 19.1 us
  // split, 14.9 us unsplit at 900 keys).
  if (Sk >= 1536 && blocks < 256)
    p.splits = std::min<int64_t>(std::min<int64_t>(cdiv(256, blocks), Sk / 256), kFrMaxSplits);
  if (p.splits > 1) p.ws_bytes = p.splits * B * Hq * Sq * (D + 4) * (int64_t)sizeof(float);
  return p;
}

template <typename T, int D>
static int launch(const FrArgs& a, int64_t blocks, hipStream_t st) {
  fa_rows<T, D><<<dim3((unsigned)blocks), kFrThreads, 0, st>>>(a);
  if (a.splits > 1)
    fa_rows_merge<T, D><<<dim3((unsigned)a.total), kFrThreads, 0, st>>>(a);
  return record_launch();
}

template <typename T>
int launch_fa_rows(const void* Q, const void* K, const void* V, void* O, int64_t B, int64_t Hq, int64_t Hkv,
                   int64_t Sq, int64_t Sk, int64_t D, const int64_t* qs, const int64_t* ks, const int64_t* vs,
                   const int64_t* os, float sm_scale, float* ws, int64_t ws_bytes, hipStream_t st) {
  const FaRowsPlan p = fa_rows_plan(B, Hq, Hkv, Sq, Sk, D, false);
  FrArgs a;
  a.Q = (const uint16_t*)Q;
  a.K = (const uint16_t*)K;
  a.V = (const uint16_t*)V;
  a.O = (uint16_t*)O;
  a.qsb = qs[0], a.qsh = qs[1], a.qss = qs[2];
  a.ksb = ks[0], a.ksh = ks[1], a.kss = ks[2];
  a.vsb = vs[0], a.vsh = vs[1], a.vss = vs[2];
  a.osb = os[0], a.osh = os[1], a.oss = os[2];
  a.Hkv = (int)Hkv;
  a.group = (int)(Hq / Hkv);
  a.Sq = (int)Sq;
  a.Sk = (int)Sk;
  a.rows = (int)(a.group * Sq);
  a.row_blocks = (int)cdiv(a.rows, kFrRows);
  a.splits = ws && ws_bytes >= p.ws_bytes ? (int)p.splits : 1;
  // whole steps per slice, and no empty slice
  a.split_keys = (int)(cdiv(cdiv(Sk, a.splits), kFrKeys) * kFrKeys);
  a.splits = (int)cdiv(Sk, a.split_keys);
  a.total = B * Hq * Sq;
  a.part = ws;
  a.stat = ws ? ws + (int64_t)a.splits * a.total * D : nullptr;
  a.c_log2 = sm_scale * kFaLog2e;
  a.thr = T::kCode == AK_F16 ? 65520.0f / fmaxf(1.0f, fabsf(sm_scale)) : INFINITY;
  const int64_t blocks = B * Hkv * a.row_blocks * a.splits;
  return D == 64 ? launch<T, 64>(a, blocks, st) : launch<T, 128>(a, blocks, st);
}

template int launch_fa_rows<TF16>(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t,
                                  int64_t, int64_t, const int64_t*, const int64_t*, const int64_t*, const int64_t*,
                                  float, float*, int64_t, hipStream_t);
template int launch_fa_rows<TBF16>(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t,
                                   int64_t, int64_t, const int64_t*, const int64_t*, const int64_t*, const int64_t*,
                                   float, float*, int64_t, hipStream_t);

}  // namespace ak

// gemm_f32.hip -- fp32 GEMM and fp32 SwiGLU gate/up on v_mfma_f32_16x16x4_f32: full fp32 products, no
// reduced-precision inputs.
//
// What bounds it: the fp32 matrix rate (157 TFLOP/s), 1/16 of the bf16 rate, so operand traffic is
// small beside the products and the design only has to keep the MFMA pipe fed:
//   * Block tile BM x BN x 32, two LDS stages filled from registers: 16-byte global loads (at any
//     alignment, see f32x4_u), 16-byte LDS writes, one barrier per tile.
//   * One 16-byte LDS read gives a lane four k of one row, the operands of four MFMAs: the four lane
//     groups of step j hold k = 4 g + j, and A and B permute k alike. A and nn.Linear-layout B rows
//     are 128 bytes with chunk c at c ^ (row & 7), the conflict-free layout of the 16-bit kernels. A
//     [K, N] B stays [k][n]: a lane reads FN consecutive n of one k, one for each of its fragments, so
//     fragment f holds columns FN i + f and a lane's results are still consecutive in n.
//   * Every 16 of k accumulate from the negated compensation of the running total and are then added
//     to it (Kahan): three VALU operations per element and 64 MFMA cycles, issued beside the next
//     fragments' MFMAs. That keeps long sums inside the 1e-4 tolerance of the op table (a plain
//     fp32 sum of K = 8192 is 4.9e-4 off).
// The order of the additions depends on k alone, so every tile size and layout gives the same bits.
//
// Measured, f32 2048^3: 306 -> 173 us (4-byte loads and LDS reads before: 56 TFLOP/s), 4096^3 98-104
// TFLOP/s; 1024^3, whose 64 tiles of 128 x 128 left most CUs idle, 154 -> 39 us on 64 x 64 tiles.
// Without the Kahan steps (a timing-only build) 2048^3 takes 17 % less. The error against 64 bits is
// 7.9e-8 (8.1e-8 before), a plain fp32 sum's 8.1e-7.
#include <limits.h>

#include "gemm_common.h"

namespace ak {

constexpr int kF32BK = 32;

// Four floats at 4-byte alignment: global loads and stores of 16 bytes take any alignment here.
typedef f32x4 f32x4_u __attribute__((aligned(4)));

// y = -c + (16 products) on entry, -c (the new negated compensation) on exit; s the running total.
__device__ __forceinline__ void kahan_step(f32x4& s, f32x4& y) {
  const f32x4 t = s + y;
  y = y - (t - s);
  s = t;
}

template <int BM, int BN, int WM, int WN, int NB, bool BT>
__global__ __launch_bounds__(WM* WN* kWave) void gemm_f32_tile(
    const float* __restrict__ A, const float* __restrict__ B0, const float* __restrict__ B1, float* __restrict__ C,
    int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles_n, int act,
    int64_t batch_a, int64_t batch_b, int64_t batch_c) {
  constexpr int BK = kF32BK, NT = WM * WN * kWave;
  constexpr int WTM = BM / WM, WTN = BN / WN, FM = WTM / 16, FN = WTN / 16;
  constexpr int ACH = BM * (BK / 4) / NT, BCH = BN * (BK / 4) / NT;  // 16-byte chunks per thread
  constexpr int BCPR = BT ? BK / 4 : BN / 4;                         // chunks per B tile row
  static_assert(ACH * NT == BM * (BK / 4) && BCH * NT == BN * (BK / 4), "tiles split evenly");
  static_assert(NB == 1 || BT, "gate/up weights are [H, D]");
  __shared__ __attribute__((aligned(16))) float sA[2][BM * BK];
  __shared__ __attribute__((aligned(16))) float sB[2][NB][BN * BK];
  if (gridDim.z > 1) {
    const int64_t z = blockIdx.z;
    A += z * batch_a;
    B0 += z * batch_b;
    C += z * batch_c;
  }
  int tm, tn;
  tile_coords(tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = lane_id(), wid = wave_id();
  const int wm = wid / WN, wn = wid % WN;
  const int fr = lane & 15, kg = lane >> 4;
  const float* Bm[2] = {B0, B1};

  // This thread's chunks. Rows past M (or N) re-read the last row; their results are not stored.
  const float* pa[ACH];
  int64_t ob[BCH];
#pragma unroll
  for (int i = 0; i < ACH; ++i) {
    const int q = tid + i * NT;
    pa[i] = A + (int64_t)min(m0 + q / (BK / 4), M - 1) * lda + (q % (BK / 4)) * 4;
  }
#pragma unroll
  for (int i = 0; i < BCH; ++i) {
    const int q = tid + i * NT;
    if constexpr (BT) ob[i] = (int64_t)min(n0 + q / BCPR, N - 1) * ldb + (q % BCPR) * 4;
    else ob[i] = (int64_t)(q / BCPR) * ldb + n0 + (q % BCPR) * 4;
  }
  f32x4 ra[ACH], rb[NB][BCH];
  auto gload = [&](int k0) {
    if (k0 + BK <= K && (BT || n0 + BN <= N)) {  // uniform: a whole tile
#pragma unroll
      for (int i = 0; i < ACH; ++i) ra[i] = *reinterpret_cast<const f32x4_u*>(pa[i] + k0);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < BCH; ++i)
          rb[b][i] = *reinterpret_cast<const f32x4_u*>(Bm[b] + ob[i] + (BT ? (int64_t)k0 : (int64_t)k0 * ldb));
    } else {  // the K tail or a ragged right edge: elements, zeros past the end
#pragma unroll
      for (int i = 0; i < ACH; ++i) {
        const int k = k0 + ((tid + i * NT) % (BK / 4)) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) ra[i][e] = k + e < K ? pa[i][k0 + e] : 0.f;
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < BCH; ++i) {
          const int q = tid + i * NT;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool in = BT ? k0 + (q % BCPR) * 4 + e < K : k0 + q / BCPR < K && n0 + (q % BCPR) * 4 + e < N;
            rb[b][i][e] = in ? Bm[b][ob[i] + (BT ? (int64_t)k0 : (int64_t)k0 * ldb) + e] : 0.f;
          }
        }
    }
  };
  // [k][n] tile: rows 4 apart, read by neighbouring lane groups, swap their 128-byte halves
  auto nn_off = [](int k, int n) { return k * BN + (n ^ (((k >> 2) & 1) << 5)); };
  auto sstore = [&](int st) {
#pragma unroll
    for (int i = 0; i < ACH; ++i) {
      const int q = tid + i * NT, row = q / (BK / 4), c = q % (BK / 4);
      *reinterpret_cast<f32x4*>(&sA[st][row * BK + (c ^ (row & 7)) * 4]) = ra[i];
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < BCH; ++i) {
        const int q = tid + i * NT, row = q / BCPR, c = q % BCPR;
        const int off = BT ? row * BK + (c ^ (row & 7)) * 4 : nn_off(row, c * 4);
        *reinterpret_cast<f32x4*>(&sB[st][b][off]) = rb[b][i];
      }
  };

  f32x4 s[NB][FM][FN], y[NB][FM][FN];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int f = 0; f < FN; ++f) s[b][i][f] = y[b][i][f] = f32x4{0.f, 0.f, 0.f, 0.f};

  // fragments of 16-deep half h of the tile in stage st
  auto load_a = [&](int st, int h, f32x4 (&fa)[FM]) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = wm * WTM + i * 16 + fr;
      fa[i] = *reinterpret_cast<const f32x4*>(&sA[st][row * BK + ((h * 4 + kg) ^ (row & 7)) * 4]);
    }
  };
  auto load_b = [&](int st, int h, f32x4 (&fb)[NB][FN]) {  // fb[b][f][j]: step j of fragment f
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if constexpr (BT) {
#pragma unroll
        for (int f = 0; f < FN; ++f) {
          const int row = wn * WTN + f * 16 + fr;
          fb[b][f] = *reinterpret_cast<const f32x4*>(&sB[st][b][row * BK + ((h * 4 + kg) ^ (row & 7)) * 4]);
        }
      } else {
        static_assert(FN == 2, "a [K, N] tile is read in pairs of columns");
        typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x2 v = *reinterpret_cast<const f32x2*>(&sB[st][b][nn_off(h * 16 + kg * 4 + j, wn * WTN + FN * fr)]);
          fb[b][0][j] = v[0];
          fb[b][1][j] = v[1];
        }
      }
    }
  };
  f32x4 fa[FM], fb[NB][FN], na[FM], nb[NB][FN];
  auto mfma_row = [&](int i) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int f = 0; f < FN; ++f)
          y[b][i][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[b][f][j], fa[i][j], y[b][i][f], 0, 0, 0);
  };
  auto kahan_row = [&](int i) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int f = 0; f < FN; ++f) kahan_step(s[b][i][f], y[b][i][f]);
  };
  // One half: each row's MFMAs beside the Kahan steps of the row before it (row 0: the last row of
  // the half before), one MFMA to three VALU instructions; left to itself the compiler sinks the
  // Kahan steps into one bunch per tile (4096^3, back to back: 1395 against 1426 us). The next half's
  // fragments load behind the first rows. cross: the next half is in the next tile, so a barrier comes
  // first (every wave has stored its share of that tile, and holds the last fragments of this one).
  auto rows = [&](int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      mfma_row(i);
      kahan_row(i > 0 ? i - 1 : FM - 1);
    }
    // keep the Kahan steps in this stretch (otherwise they sink to their first use, after the barrier)
#pragma unroll
    for (int i = i0; i < i1; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int f = 0; f < FN; ++f) asm volatile("" : "+v"(y[b][i > 0 ? i - 1 : FM - 1][f]));
#pragma unroll
    for (int i = 0; i < (i1 - i0) * 4 * NB * FN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto half = [&](int nst, int nh, bool cross) {
    rows(0, FM / 2);
    if (cross) dma_barrier<63>();
    load_a(nst, nh, na);
    load_b(nst, nh, nb);
    __builtin_amdgcn_sched_barrier(0);
    rows(FM / 2, FM);
#pragma unroll
    for (int i = 0; i < FM; ++i) fa[i] = na[i];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int f = 0; f < FN; ++f) fb[b][f] = nb[b][f];
  };

  // Tile kt + 1 goes to LDS halfway through tile kt, a whole tile after its loads were issued; the
  // stage it overwrites was last read before the previous barrier.
  const int KT = (K + BK - 1) / BK;
  gload(0);
  sstore(0);
  if (KT > 1) gload(BK);
  dma_barrier<63>();
  load_a(0, 0, fa);
  load_b(0, 0, fb);
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    half(cur, 1, false);
    if (kt + 1 < KT) sstore(cur ^ 1);
    if (kt + 2 < KT) gload((kt + 2) * BK);
    half(cur ^ 1, 0, true);  // after the last tile: fragments nobody uses
  }
  kahan_row(FM - 1);

  // A total that became infinite (an infinite product, an overflow) turns to NaN at the step after it,
  // inf - inf, where a plain sum stays infinite. So a block that ends with a NaN adds its products again
  // without compensation and takes those sums for its NaN elements. Finite products pay for the test
  // (us, without / with: 2048^3 170.6 / 172.2, 4096^3 1334 / 1342), a NaN or infinity anywhere for a second
  // pass (2048^3 320). Bounding the compensation at every step instead (one v_med3_f32 an element and
  // 16 of k) costs every product as much as a step of its own: 2048^3 193, 4096^3 1514.
  bool nan = false;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) nan |= s[b][i][f][e] != s[b][i][f][e];
  float* flag = &sA[0][0];  // past the last barrier no wave uses what it reads of the stages
  if (tid == 0) *flag = 0.f;
  __syncthreads();
  if (nan) *flag = 1.f;
  __syncthreads();
  if (*flag != 0.f) {  // uniform over the block
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int f = 0; f < FN; ++f) y[b][i][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < KT; ++kt) {
      gload(kt * BK);
      __syncthreads();
      sstore(0);
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        load_a(0, h, fa);
        load_b(0, h, fb);
#pragma unroll
        for (int i = 0; i < FM; ++i) mfma_row(i);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int f = 0; f < FN; ++f)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (s[b][i][f][e] != s[b][i][f][e]) s[b][i][f][e] = y[b][i][f][e];
  }

  // Lane group g = lane / 16 holds, of row m, columns 16 f + 4 g + v ([N, K] B) or FN (4 g + v) + f
  // ([K, N] B): either way FN groups of four consecutive columns.
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + wm * WTM + i * 16 + fr;
    if (m >= M) continue;
#pragma unroll
    for (int t = 0; t < FN; ++t) {
      const int n = n0 + wn * WTN + (BT ? t * 16 + kg * 4 : FN * 4 * kg + 4 * t);
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int f = BT ? t : (4 * t + e) % FN, v = BT ? e : (4 * t + e) / FN;
        if constexpr (NB == 1) {
          o[e] = s[0][i][f][v];
        } else {
          const float g = s[0][i][f][v], u = s[1][i][f][v];
          switch (act) {
            case kEpiSilu: o[e] = gate_up<TF32, kEpiSilu>(g, u); break;
            case kEpiGelu: o[e] = gate_up<TF32, kEpiGelu>(g, u); break;
            case kEpiRelu2: o[e] = gate_up<TF32, kEpiRelu2>(g, u); break;
            default: o[e] = gate_up<TF32, kEpiNone>(g, u); break;
          }
        }
      }
      float* c = C + (int64_t)m * ldc + n;
      if (n + 3 < N) {
        *reinterpret_cast<f32x4_u*>(c) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = o[e];
      }
    }
  }
}

// Tile choice: the rounds of 256 CUs a tiling takes, times its tile's MFMA work. The small tile pays
// about 15 % more per flop (half the reuse per LDS read and barrier).
static bool small_tile32(int64_t M, int64_t N, int64_t batch, int bn_big) {
  const int64_t big = cdiv(cdiv(M, 128) * cdiv(N, bn_big) * batch, 256) * 4;
  const int64_t small = cdiv(cdiv(M, 64) * cdiv(N, bn_big / 2) * batch, 256);
  return 1.15 * (double)small < (double)big;
}

// Few rows (gemm_small) instead of tiles: not for wide, shallow or very wide products of more than 32
// (16) rows, whose tiles fill the chip (us, tiles / gemm_small: 48 x 50257 x 768 84 / 108, 33 x 14976 x 179
// 10.8 / 15.1, gate/up 64 x 5120 -> 13824 264 / 317; but 64 x 11008 x 4096 142 / 123, 64 x 4096 x 4096
// 142 / 38).
static bool small_rows32(int64_t M, int64_t N, int64_t K, int nb) {
  if (M > kSmallM || K == 0 || N > small_max_n(nb)) return false;
  if (M > 32 && N > 4096 && (N > 12288 || K < 1024)) return false;
  return !(M > 16 && N > 8192 && K < 512);
}

template <int BM, int BN, int WM, int WN, int NB, bool BT>
static void launch_tile32(const void* A, const void* B0, const void* B1, void* C, int64_t M, int64_t N, int64_t K,
                          int64_t lda, int64_t ldb, int64_t ldc, int act, hipStream_t s, int batch, int64_t ba,
                          int64_t bb, int64_t bc) {
  const int tiles_m = (int)cdiv(M, BM), tiles_n = (int)cdiv(N, BN);
  gemm_f32_tile<BM, BN, WM, WN, NB, BT><<<dim3(tiles_m * tiles_n, 1, batch), WM * WN * kWave, 0, s>>>(
      (const float*)A, (const float*)B0, (const float*)B1, (float*)C, (int)M, (int)N, (int)K, lda, ldb, ldc, tiles_m,
      tiles_n, act, ba, bb, bc);
}

int launch_gemm32(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda,
                  int64_t ldb, int64_t ldc, bool bt, hipStream_t s, int batch, int64_t batch_a, int64_t batch_b,
                  int64_t batch_c) {
  if (small_rows32(M, N, K, 1)) {
    EpiArgs ep;
    ep.batch = batch;
    ep.batch_a = batch_a;
    ep.batch_b = batch_b;
    ep.batch_c = batch_c;
    return launch_gemm_small<TF32, 1, kEpiStore>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, bt, s, ep);
  }
#define AK_T32(BM, WN, BT) \
  launch_tile32<BM, BM, 2, WN, 1, BT>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, 0, s, batch, batch_a, batch_b, batch_c)
  if (small_tile32(M, N, batch, 128)) {
    if (bt) AK_T32(64, 2, true);
    else AK_T32(64, 2, false);
  } else {
    if (bt) AK_T32(128, 4, true);
    else AK_T32(128, 4, false);
  }
#undef AK_T32
  return record_launch();
}

int launch_gate_up32(const void* x, const void* wg, const void* wu, void* h, int64_t M, int64_t H, int64_t D,
                     int epi, hipStream_t s) {
  if (small_rows32(M, H, D, 2)) {
    const EpiArgs ep;
    switch (epi) {
      case kEpiSilu: return launch_gemm_small<TF32, 2, kEpiSilu>(x, wg, wu, h, M, H, D, D, D, H, true, s, ep);
      case kEpiGelu: return launch_gemm_small<TF32, 2, kEpiGelu>(x, wg, wu, h, M, H, D, D, D, H, true, s, ep);
      case kEpiRelu2: return launch_gemm_small<TF32, 2, kEpiRelu2>(x, wg, wu, h, M, H, D, D, D, H, true, s, ep);
      default: return launch_gemm_small<TF32, 2, kEpiNone>(x, wg, wu, h, M, H, D, D, D, H, true, s, ep);
    }
  }
  if (small_tile32(M, H, 1, 64))
    launch_tile32<64, 32, 2, 2, 2, true>(x, wg, wu, h, M, H, D, D, D, H, epi, s, 1, 0, 0, 0);
  else
    launch_tile32<128, 64, 2, 4, 2, true>(x, wg, wu, h, M, H, D, D, D, H, epi, s, 1, 0, 0, 0);
  return record_launch();
}

}  // namespace ak

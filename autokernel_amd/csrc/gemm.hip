// gemm.hip -- LDS-tiled MFMA GEMM for gfx950 (f16 / bf16 in, fp32 accumulate), the dual-B
// SwiGLU gate/up kernel built on it, and the GEMM entry points (fp32 kernels: gemm_f32.hip).
//
// f16 / bf16 design
//   * Block tile BM x BN (BN per B matrix; NB = 1 plain GEMM, NB = 2 gate and up sharing the A
//     tile). WM x WN waves; each wave owns a (BM/WM) x (BN/WN) sub-tile per B matrix made of
//     16x16 v_mfma_f32_16x16x32_{f16,bf16} tiles. The MFMA is issued with B as the "A" operand,
//     so a lane's accumulator holds four consecutive C columns of one row (8-byte stores).
//   * Main kernel (gemm_dma, K-contiguous B = nn.Linear weights, K % 64 == 0): operands reach LDS
//     by LDS DMA, two or three 64-deep stages (four 32-deep ones when the grid under-fills the
//     chip), so one or two tiles stream in while one is multiplied. Inside a tile the next
//     k-step's fragments load from LDS while the current MFMAs run, and the barrier that retires
//     a stage sits between the two halves of a k-step's MFMAs.
//   * Fallback kernel (gemm_mfma: any alignment, odd K, strided or [K, N] B): register-staged
//     loads into two LDS stages of [rows][64], chunks XOR-swizzled; [K, N] B is transposed in
//     registers on its way to LDS (8x8 blocks rebuilt as K-contiguous rows with v_perm_b32).
//   * Tile order is XCD-aware: hardware hands block i to XCD i % 8, so consecutive logical tiles
//     are given to one XCD and grouped along M to share A and B in that XCD's L2.
#include <limits.h>

#include "gemm_common.h"

namespace ak {

constexpr int kBK = 64;           // k extent of one LDS tile
constexpr int kKC = kBK / 8;      // 16-byte chunks per tile row

// Physical chunk of logical chunk c in row `row`. Rows r and r + 8 get different patterns, so
// both the 16-row fragment reads and the transposed [K,N] writes (rows 8 apart) are conflict-free.
__device__ __forceinline__ int swz(int row, int c) { return c ^ ((row ^ (row >> 3)) & 7); }
// element offset of chunk c of row `row` in a [rows][64] tile
__device__ __forceinline__ int lds_off(int row, int c) { return row * kBK + swz(row, c) * 8; }

// The LDS-DMA kernel's MFMA: v_mfma_f32_16x16x32 (f32x4 accumulators), 8 consecutive k of one row
// per lane. (32x32x16 fragments were measured 4-10 % slower on every workload.)
template <int MF>
struct MfmaAcc {
  static_assert(MF == 16, "the LDS-DMA kernel uses 16x16x32 fragments");
  using type = f32x4;
};
template <typename T, int MF>
__device__ __forceinline__ typename MfmaAcc<MF>::type mfma_tile(const u32x4& a, const u32x4& b,
                                                                const typename MfmaAcc<MF>::type& c) {
  return mfma16x16x32<T>(a, b, c);
}

// Load 8 consecutive k of one row of a K-contiguous matrix (row stride ld). Out-of-range rows or
// k give zeros. VEC: K, ld and the base are multiples of 8 elements / 16 bytes.
template <bool VEC>
__device__ __forceinline__ u32x4 load_kchunk(const uint16_t* __restrict__ p, int64_t ld, int row, int rows,
                                             int k, int K) {
  if constexpr (VEC) {
    if (row < rows && k < K) return ld16(p + (int64_t)row * ld + k);
    return u32x4{0u, 0u, 0u, 0u};
  } else {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < rows) {
      const uint16_t* q = p + (int64_t)row * ld;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t h = (k + e < K) ? q[k + e] : 0u;
        v[e >> 1] |= h << ((e & 1) * 16);
      }
    }
    return v;
  }
}

// gemm_small's order of the sums (N <= 4096), for tiles of a batch of such products: slice i is k-groups i,
// i + 16, ..., and the slices' sums are added as a tree over 16 waves adds them. With the slices visited in
// bit-reversed order each pair of the tree is complete before the next begins, so four held tiles are enough.
// Fewer groups than slices leave the upper slices empty: only the tree's levels below those are walked.
struct SliceWalk {
  int groups, levels, g = 0, i = 0;  // i: position of g's slice (2^levels: past the end)
  __device__ __forceinline__ explicit SliceWalk(int n) : groups(n), levels(n > 8 ? 4 : n > 4 ? 3 : n > 2 ? 2 : n > 1 ? 1 : 0) {}
  __device__ __forceinline__ bool done() const { return i >> levels; }
  __device__ __forceinline__ void step() {
    for (g += 16; g >= groups && !done();) {
      ++i;
      g = (int)((__builtin_bitreverse32((unsigned)i) >> 1) >> (31 - levels));
    }
  }
};
// The slice at position i is in acc: hold it (acc starts the next) or add it to the held left halves it ends.
// Level d of part holds 2^d slices. (With part in LDS, or with the walk unrolled, the tiles were slower.)
template <int FM, int FN>
__device__ __forceinline__ void end_slice(int i, int levels, f32x4 (&part)[4][FM][FN], f32x4 (&acc)[FM][FN]) {
  bool held = false;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    if (held || d >= levels) continue;
    held = ((i >> d) & 1) == 0;  // uniform
#pragma unroll
    for (int x = 0; x < FM; ++x)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if (held) {
          part[d][x][j] = acc[x][j];
          acc[x][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        } else {
          acc[x][j] = part[d][x][j] + acc[x][j];
        }
      }
  }
}

// --------------------------------------------------------------------------------------------
// The f16 / bf16 kernel. SL: 0, or the depth of a k-group (32 or 64) summed in gemm_small's order.
// --------------------------------------------------------------------------------------------
template <typename T, bool BT, bool VEC, int BM, int BN, int WM, int WN, int NB, int EPI, int SL = 0>
__global__ __launch_bounds__(WM* WN* kWave) void gemm_mfma(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1,
    uint16_t* __restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    int tiles_m, int tiles_n, EpiArgs ep) {
  constexpr int kThreads = WM * WN * kWave;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  constexpr int A_CH = BM * kKC / kThreads;  // A chunks per thread
  static_assert(BM * kKC % kThreads == 0, "A tile must split evenly");
  constexpr int BT_CH = (BN * kKC + kThreads - 1) / kThreads;      // [N,K] B chunks per thread
  constexpr int BN_UNITS = (kBK / 4) * (BN / 8);                   // [K,N] B 4x8 units per matrix
  constexpr int BN_U = (BN_UNITS + kThreads - 1) / kThreads;

  __shared__ __attribute__((aligned(16))) uint16_t sA[2][BM * kBK];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][NB][BN * kBK];
  if constexpr (SL != 0) {
    if (skip_item(ep)) return;
  }
  batch_bases(A, B0, C, ep);

  int tm, tn;
  tile_coords(tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wid = wave_id();
  const int wm = wid / WN, wn = wid % WN;
  const uint16_t* Bm[2] = {B0, B1};

  // ---- global -> register staging ----
  u32x4 ra[A_CH];
  u32x4 rbt[NB][BT ? BT_CH : 1];
  u32x4 rbn[BT ? 1 : BN_U][4];

  // The tile's halves of 32 are k0 .. and k1 .. (k0 + 32 unless SL is 32).
  auto gload = [&](int k0, int k1) {
    auto at = [&](int p) { return SL == 32 && p >= 32 ? k1 + p - 32 : k0 + p; };
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int q = tid + i * kThreads;
      const int row = q / kKC, c = q % kKC;
      ra[i] = load_kchunk<VEC>(A, lda, m0 + row, M, at(c * 8), K);
    }
    if constexpr (BT) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < BT_CH; ++i) {
          const int q = tid + i * kThreads;
          const int row = q / kKC, c = q % kKC;
          if (q < BN * kKC) rbt[b][i] = load_kchunk<VEC>(Bm[b], ldb, n0 + row, N, at(c * 8), K);
        }
    } else {
#pragma unroll
      for (int i = 0; i < BN_U; ++i) {
        const int u = tid + i * kThreads;
        // consecutive lanes take consecutive 8-column groups of the same 4 k-rows (coalesced)
        const int ng = u % (BN / 8), kq = u / (BN / 8);
        if (u < BN_UNITS) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int k = at(kq * 4) + r;
            const int n = n0 + ng * 8;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (k < K) {
              const uint16_t* p = B0 + (int64_t)k * ldb + n;
              if constexpr (VEC) {
                if (n < N) v = ld16(p);
              } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  const uint32_t h = (n + e < N) ? p[e] : 0u;
                  v[e >> 1] |= h << ((e & 1) * 16);
                }
              }
            }
            rbn[i][r] = v;
          }
        }
      }
    }
  };
  auto sstore = [&](int st) {
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int q = tid + i * kThreads;
      const int row = q / kKC, c = q % kKC;
      *reinterpret_cast<u32x4*>(&sA[st][lds_off(row, c)]) = ra[i];
    }
    if constexpr (BT) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < BT_CH; ++i) {
          const int q = tid + i * kThreads;
          const int row = q / kKC, c = q % kKC;
          if (q < BN * kKC) *reinterpret_cast<u32x4*>(&sB[st][b][lds_off(row, c)]) = rbt[b][i];
        }
    } else {
#pragma unroll
      for (int i = 0; i < BN_U; ++i) {
        const int u = tid + i * kThreads;
        const int ng = u % (BN / 8), kq = u / (BN / 8);
        if (u < BN_UNITS) {
          u32x2 t[8];
          transpose4x8(rbn[i], t);
#pragma unroll
          for (int n = 0; n < 8; ++n)
            *reinterpret_cast<u32x2*>(&sB[st][0][lds_off(ng * 8 + n, kq >> 1) + (kq & 1) * 4]) = t[n];
        }
      }
    }
  };

  f32x4 acc[NB][FM][FN];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int groups = SL ? (K + SL - 1) / (SL ? SL : 1) : 0;
  const int KT = SL == 32 ? (groups + 1) / 2 : (K + kBK - 1) / kBK;
  f32x4 part[4][SL ? FM : 1][SL ? FN : 1];
  SliceWalk fetch(groups), use(groups);
  auto take = [&]() {  // the next group's k; past the last one K, whose loads are zeros
    const int k = fetch.done() ? K : fetch.g * SL;
    fetch.step();
    return k;
  };
  auto load_tile = [&](int kt) {
    if constexpr (SL) {
      const int k0 = take();
      gload(k0, SL == 32 ? take() : k0 + 32);
    } else {
      gload(kt * kBK, kt * kBK + 32);
    }
  };
  load_tile(0);
  sstore(0);
  __syncthreads();

  const int fr = lane & 15;        // fragment row owned by this lane
  const int fc = lane >> 4;        // 8-element k group inside a 32-k step
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < KT) load_tile(kt + 1);
#pragma unroll
    for (int s = 0; s < kBK / 32; ++s) {
      u32x4 fa[FM], fb[NB][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int row = wm * WTM + i * 16 + fr;
        fa[i] = *reinterpret_cast<const u32x4*>(&sA[cur][lds_off(row, s * 4 + fc)]);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int row = wn * WTN + j * 16 + fr;
          fb[b][j] = *reinterpret_cast<const u32x4*>(&sB[cur][b][lds_off(row, s * 4 + fc)]);
        }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[b][i][j] = mfma16x16x32<T>(fb[b][j], fa[i], acc[b][i][j]);
      if constexpr (SL != 0) {
        if (SL == 32 || s == 1) {
          int i = use.i;
          use.step();
          for (; i < use.i; ++i) end_slice<FM, FN>(i, use.levels, part, acc[0]);
        }
      }
    }
    if (kt + 1 < KT) sstore(cur ^ 1);
    __syncthreads();
  }

  // ---- epilogue: lane holds C[m][n .. n+3] for each (i, j) ----
  tile_epilogue<T, NB, EPI, VEC, FM, FN>(C, B1, ldc, M, N, m0 + wm * WTM + fr, n0 + wn * WTN + fc * 4, acc, ep);
}

// --------------------------------------------------------------------------------------------
// The f16 / bf16 kernel for K-contiguous B ([N, K], nn.Linear weights) with K % 64 == 0.
// Tiles move global -> LDS with gfx950's LDS DMA (global_load_lds_dwordx4): no staging registers
// and no LDS store instructions. One DMA instruction writes 64 lanes x 16 bytes = 1 KB of
// consecutive tile rows; each lane fetches the logical chunk that the XOR swizzle maps to its
// physical slot. Rows past M / N are clamped to the last row (their results are never stored).
// gfx950 serves a 64-lane ds_read_b128 in 8-lane phases, so the swizzles put the 8 rows of a phase
// in 8 distinct 16-byte bank slots (measured for 128-byte rows: SQ_LDS_BANK_CONFLICT 0 with
// chunk c ^ (row & 7), 50% with an extra row-bit-3 term, 75% unswizzled).
// --------------------------------------------------------------------------------------------
// LDS-DMA helpers (lds_void, wait_vmcnt, dma_barrier) live in ak_common.h.

// The same transfer as inline assembly. The compiler then does not track it: its wait-count pass
// inserts no waits for it (a conservative full wait at a loop head otherwise drains the whole
// four-stage pipeline once per iteration), and every wait is the caller's explicit vmcnt. M0
// holds the wave-uniform LDS destination. It is an input operand bound to M0 ("{m0}"), so the
// compiler writes M0 itself and knows its value; the statement changes no register behind the
// compiler's back. One wait state separates the M0 write from the load.
__device__ __forceinline__ void dma16_asm(const char* base, uint32_t off, uint16_t* lds_row_base) {
  const uint32_t lds = (uint32_t)(uintptr_t)(lds_void*)lds_row_base;
  asm volatile(
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(off), "s"(base), "{m0}"(lds)
      : "memory");
}

// Multi-stage variant: NS LDS stages of BKD-deep tiles (BKD 64: 128-byte rows, chunk c of row r
// at c ^ (r & 7), 8 rows per DMA instruction; BKD 32: 64-byte rows, chunk c at c ^ ((r >> 2) & 1),
// 16 rows per instruction; either way the 8 rows of one ds_read_b128 phase hit 8 distinct 16-byte
// bank slots). NS - 1 tiles are in flight while one is multiplied. Tile t lives in stage t % NS;
// the loop runs in groups of NS tiles with a uniform guard on the tail.
template <int BKD>
struct DmaGeom;
template <>
struct DmaGeom<64> {
  static constexpr int RPI = 8;  // rows per 1 KB DMA instruction
  __device__ static __forceinline__ int swz(int r, int c) { return c ^ (r & 7); }
};
template <>
struct DmaGeom<32> {
  static constexpr int RPI = 16;
  __device__ static __forceinline__ int swz(int r, int c) { return c ^ ((r >> 2) & 1); }
};

// [K, N] B (N contiguous, torch.matmul's B) is staged as [k][n] tile rows. The MFMA operand needs
// 8 consecutive k of one n per lane: two ds_read_b64_tr_b16 each give 4. That instruction
// transposes across each group of 16 lanes: output lane i, element e = element (i % 4) of source
// lane (i / 4 + 4 e); so source lane j addresses B[k0 + j / 4][n0 + 4 (j % 4)] and output lane i
// receives B[k0 + e][n0 + i]. 16-byte chunk c of tile row k is stored at c ^ bkn_swz<BN>(k): the 16
// rows of one tr read (4 per lane group) land on distinct banks for lane groups {0,1}, {2,3},
// {0,2} and {1,3}.
// A 64-element tile row (BN = 64) has 8 chunks and 128 bytes, so rows r and r + 2 share banks: the
// pattern 2 ((k >> 1) & 1) + 4 (((k >> 3) ^ (k >> 4)) & 1) keeps each read's chunk pair inside the row
// and gives rows {0, 2, 8, 10}, {0, 2, 16, 18} and {8, 10, 24, 26} distinct chunk pairs (rows + 4,
// the second read, share the pattern).
template <int BN>
__device__ __forceinline__ int bkn_swz(int k) {
  if constexpr (BN == 64) return 2 * (((k >> 1) & 1) + 2 * (((k >> 3) ^ (k >> 4)) & 1));
  else return 2 * ((k & 3) + 4 * (((k >> 3) ^ (k >> 4)) & 1));
}

typedef short gemm_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 lds_tr16(const uint16_t* p) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gemm_s16x4*)(p)));
}

// B-side DMA geometry: BKN (B is [K, N]) stages BKD rows of BN elements, else BN rows of BKD.
template <int BN, int BKD, bool BKN>
struct DmaB {
  static constexpr int kRowElems = BKN ? BN : BKD;
  static constexpr int RPI = 512 / kRowElems;    // tile rows per 1 KB transfer
  static constexpr int kRows = BKN ? BKD : BN;   // tile rows per stage
};

// SL: the k-tiles are the groups of gemm_small's order.
template <typename T, int BM, int BN, int WM, int WN, int NB, int BKD, int NS, bool BKN, int MF, bool SL>
__device__ __forceinline__ void gemm_dma_ns_kloop(
    typename MfmaAcc<MF>::type (&acc)[NB][BM / WM / MF][BN / WN / MF], const uint16_t* A, const uint16_t* B0,
    const uint16_t* B1, const uint32_t* oa, const uint32_t* ob, uint32_t kb_step_b, int K, int wid,
    int wm, int wn, int lane, uint16_t* s0, uint16_t* s1, uint16_t* s2, uint16_t* s3) {
  using G = DmaGeom<BKD>;
  using GB = DmaB<BN, BKD, BKN>;
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / MF, FN = WTN / MF;
  constexpr int A_INS = BM / G::RPI / NW;
  constexpr int B_INS = GB::kRows / GB::RPI / NW;
  constexpr int INS = A_INS + NB * B_INS;
  constexpr int H = FM / 2;
  constexpr int KS = 32;  // k per MFMA
  constexpr int STEPS = BKD / KS;         // k-steps per tile
  static_assert(NS >= 2 && NS <= 4, "stages");
  const uint16_t* Bm[2] = {B0, B1};
  // fragment row (lane % MF) and 16-byte k chunk (lane / MF) of this lane
  const int fr = lane & (MF - 1), fc = lane / MF;
  uint16_t* const st[4] = {s0, s1, s2, s3};

  const int KT = K / BKD;
  f32x4 part[4][SL ? FM : 1][SL ? FN : 1];
  SliceWalk fetch(KT), use(KT);
  auto issue = [&](int kt, uint16_t* sp) {
    if constexpr (SL) {  // issues come in the tiles' order; past the end the last one again
      kt = fetch.g;
      SliceWalk n = fetch;
      n.step();
      if (!n.done()) fetch = n;
    }
    const uint32_t kb = 2u * (uint32_t)(kt * BKD);
    const uint32_t kbb = BKN ? (uint32_t)kt * kb_step_b : kb;
#pragma unroll
    for (int i = 0; i < A_INS; ++i)
      dma16_asm(reinterpret_cast<const char*>(A), oa[i] + kb, sp + (i * NW + wid) * 512);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < B_INS; ++i)
        dma16_asm(reinterpret_cast<const char*>(Bm[b]), ob[i] + kbb, sp + (BM + b * BN) * BKD + (i * NW + wid) * 512);
  };
  u32x4 fa[FM], fb[NB][FN], fbn[NB][FN];
  auto frag = [&](const uint16_t* base, int row, int s) -> u32x4 {
    return *reinterpret_cast<const u32x4*>(&base[row * BKD + G::swz(row, s * (KS / 8) + fc) * 8]);
  };
  auto load_a = [&](const uint16_t* sp, int s, int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i) fa[i] = frag(sp, wm * WTM + i * MF + fr, s);
  };
  auto load_b = [&](const uint16_t* sp, int s, u32x4 (*dst)[FN]) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if constexpr (BKN) {
          // k = 32 s + 8 (lane / 16) + 0..3 and + 4..7 for n = wn * WTN + 16 j + lane % 16
          const uint16_t* bs = sp + (BM + b * BN) * BKD;
          const int row = s * 32 + 8 * fc + (fr >> 2);
          const int col = wn * WTN + j * 16 + 4 * (fr & 3);
          const uint16_t* p = bs + row * BN + (((col >> 3) ^ bkn_swz<BN>(row)) * 8) + (col & 7);
          const u32x2 lo = lds_tr16(p);
          const u32x2 hi = lds_tr16(p + 4 * BN);  // rows + 4 share the swizzle
          dst[b][j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        } else {
          dst[b][j] = frag(sp + (BM + b * BN) * BKD, wn * WTN + j * MF + fr, s);
        }
      }
  };
  auto mfma_rows = [&](int i0, int i1) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = i0; i < i1; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[b][i][j] = mfma_tile<T, MF>(fb[b][j], fa[i], acc[b][i][j]);
  };
  // One k-step: first half of the MFMAs; at a tile's last step (cross) wait until the next tile
  // has landed (NS - 2 later tiles may still be in flight), barrier (every wave holds this tile's
  // fragments, so its stage is free) and refill the stage with tile refill_kt (clamped: past the
  // end it re-fetches the last tile into a stage nobody reads again); the next step's fragments
  // load around the second half.
  auto kstep = [&](const uint16_t* nsp, int ns, bool cross, uint16_t* rsp, int refill_kt) {
    mfma_rows(0, H);
    __builtin_amdgcn_sched_barrier(0);
    if (cross) {
      dma_barrier<(NS - 2) * INS>();
      issue(refill_kt, rsp);
    }
    load_a(nsp, ns, 0, H);
    load_b(nsp, ns, fbn);
    __builtin_amdgcn_sched_barrier(0);
    mfma_rows(H, FM);
    __builtin_amdgcn_sched_barrier(0);
    load_a(nsp, ns, H, FM);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[b][j] = fbn[b][j];
  };
#pragma unroll
  for (int i = 0; i < NS; ++i) issue(min(i, KT - 1), st[i]);
  dma_barrier<(NS - 1) * INS>();
  load_a(s0, 0, 0, FM);
  load_b(s0, 0, fb);
  if constexpr (SL) {
    static_assert(NB == 1 && NS == 4, "slices of one product, in four stages");
    constexpr int kStage = (BM + BN) * BKD;
    // Not unrolled over the stages (which are one array): the longer code cost more to fetch than it saved (us,
    // unrolled / so: 128 x [64 x 64 x 512] 10.3 / 8.5, 256 x [32 x 1024 x 512] 80 / 73; 128 x [64 x 1024 x 1024] 73 / 76).
#pragma unroll 1
    for (int t = 0; t < KT; ++t) {
      uint16_t* const cur = s0 + (t & 3) * kStage;
      uint16_t* const nxt = s0 + ((t + 1) & 3) * kStage;
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        if (s + 1 < STEPS) kstep(cur, s + 1, false, cur, 0);
        else kstep(nxt, 0, true, cur, 0);
      }
      int i = use.i;
      use.step();
#pragma unroll 1
      for (; i < use.i; ++i) end_slice<FM, FN>(i, use.levels, part, acc[0]);
    }
  } else {
    for (int kt = 0; kt < KT; kt += NS) {
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int t = kt + u;
        if (t < KT) {  // uniform over the block
#pragma unroll
          for (int s = 0; s < STEPS; ++s) {
            if (s + 1 < STEPS) kstep(st[u], s + 1, false, st[u], 0);
            else kstep(st[(u + 1) % NS], 0, true, st[u], min(t + NS, KT - 1));
          }
        }
      }
    }
  }
  wait_vmcnt<0>();  // no DMA may still target this block's LDS when its waves end
}

// Store a block's tile by whole rows through LDS, for a C with rows at odd element offsets (an odd ldc,
// e.g. a 50257-column vocabulary projection). From the fragments a store instruction writes 64 bytes
// of each of 16 rows; where those start off a dword they cost twice the requests of dword-aligned
// ones, while a wave that stores whole rows of the tile pays for a row's two ends only (f16, us, from
// the fragments / by rows / an even ldc: 2048x50257x768 224 / 199 / 196, 8192x50257x768 838 / 761 / 732;
// an even ldc is 2 % slower by rows). The tile's halves of BM / 2 rows go to s0 and s1, two of the
// stages (free once every wave is past the k-loop), 16-byte chunk c of row r at c ^ (r & 7): the 8 lanes
// of a write (8 rows) or a read (8 chunks) hit distinct bank slots.
template <typename T, int BM, int BN, int NW, int FM, int FN>
__device__ __forceinline__ void store_tile_rows(uint16_t* __restrict__ C, int64_t ldc, int M, int N, int m0, int n0,
                                                int row0, int col0, const f32x4 (&acc)[FM][FN], uint16_t* s0, uint16_t* s1) {
  constexpr int CPR = BN / 8;  // chunks per row
  static_assert(BM * CPR % (NW * kWave) == 0 && CPR % 8 == 0, "whole rows of chunks over the block");
  const int lane = lane_id(), fr = lane & 15, fc = lane >> 4;
  const auto row = [&](int r) { return (r < BM / 2 ? s0 : s1) + (r % (BM / 2)) * BN; };
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int r = row0 + i * 16 + fr;
    uint32_t lo[FN], hi[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      lo[j] = (uint32_t)T::from_f(acc[i][j][0]) | ((uint32_t)T::from_f(acc[i][j][1]) << 16);
      hi[j] = (uint32_t)T::from_f(acc[i][j][2]) | ((uint32_t)T::from_f(acc[i][j][3]) << 16);
    }
#pragma unroll
    for (int j = 0; j + 1 < FN; j += 2) {
      regroup8(lo[j], lo[j + 1]);
      regroup8(hi[j], hi[j + 1]);
      const int c = col0 / 8 + j * 2 + fc;
      *reinterpret_cast<u32x4*>(row(r) + (c ^ (r & 7)) * 8) = u32x4{lo[j], hi[j], lo[j + 1], hi[j + 1]};
    }
    if constexpr (FN % 2 == 1) {
      const int c = col0 / 8 + (FN - 1) * 2 + fc / 2;
      *reinterpret_cast<u32x2*>(row(r) + (c ^ (r & 7)) * 8 + (fc & 1) * 4) = u32x2{lo[FN - 1], hi[FN - 1]};
    }
  }
  __syncthreads();
#pragma unroll 4
  for (int q = threadIdx.x; q < BM * CPR; q += NW * kWave) {
    const int r = q / CPR, c = q % CPR;
    const u32x4 o = *reinterpret_cast<const u32x4*>(row(r) + (c ^ (r & 7)) * 8);
    if (m0 + r < M) store_cols<true, 8>(C + (int64_t)(m0 + r) * ldc + n0 + c * 8, N - n0 - c * 8, o);
  }
}

template <typename T, int BM, int BN, int WM, int WN, int NB, int EPI, int BKD, int NS, bool BKN, int MF, int OCC, bool SL>
__global__ __launch_bounds__(WM* WN* kWave, OCC* WM* WN / 4) void gemm_dma(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1,
    uint16_t* __restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    int tiles_m, int tiles_n, EpiArgs ep) {
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / MF, FN = WTN / MF;  // MFMA fragments per wave along M and N
  constexpr int RPI = DmaGeom<BKD>::RPI;  // tile rows per DMA instruction (1 KB)
  using GB = DmaB<BN, BKD, BKN>;
  constexpr int A_INS = BM / RPI / NW;  // DMA instructions per wave per tile for A
  constexpr int B_INS = GB::kRows / GB::RPI / NW;  // ... per B matrix
  static_assert(A_INS * RPI * NW == BM && B_INS * GB::RPI * NW == GB::kRows, "tile rows split over waves");
  static_assert(4 * (A_INS + NB * B_INS) < 64, "outstanding DMA fits vmcnt");
  static_assert(FM % 2 == 0, "two MFMA halves per k-step");
  constexpr int kStage = (BM + NB * BN) * BKD;  // elements per stage
  __shared__ __attribute__((aligned(1024))) uint16_t sS0[SL ? NS * kStage : kStage];
  __shared__ __attribute__((aligned(1024))) uint16_t sS1s[SL ? 1 : kStage];
  __shared__ __attribute__((aligned(1024))) uint16_t sS2s[!SL && NS > 2 ? kStage : 1];
  __shared__ __attribute__((aligned(1024))) uint16_t sS3s[!SL && NS > 3 ? kStage : 1];
  uint16_t* const sS1 = SL ? sS0 + kStage : sS1s;
  uint16_t* const sS2 = SL ? sS0 + 2 * kStage : sS2s;
  uint16_t* const sS3 = SL ? sS0 + 3 * kStage : sS3s;

  if constexpr (EPI == kEpiPartial) {
    const int z = (int)blockIdx.y;  // K slice
    A += z * ep.split_a;
    B0 += z * ep.split_b;
    C += 2 * z * ep.split_c;  // fp32 workspace addressed in 16-bit units
  }
  batch_bases(A, B0, C, ep);
  int tm, tn;
  tile_coords(tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = lane_id();
  const int wid = __builtin_amdgcn_readfirstlane(wave_id());  // wave-uniform: LDS bases in SGPRs
  const int wm = wid / WN, wn = wid % WN;
  const int r_in = lane / (64 / RPI), pc = lane % (64 / RPI);

  // Per-lane byte offsets (fixed over k; the host guarantees M * lda and N * ldb elements fit
  // 31 bits, so bytes fit 32) of the row and chunk each DMA instruction fetches: physical chunk pc
  // of a row holds logical chunk swz(row, pc) (each XOR pattern is its own inverse).
  uint32_t oa[A_INS];
#pragma unroll
  for (int i = 0; i < A_INS; ++i) {
    const int row = (i * NW + wid) * RPI + r_in;
    const int lc = DmaGeom<BKD>::swz(row, pc);
    oa[i] = 2u * (uint32_t)(min(m0 + row, M - 1) * (int)lda + lc * 8);
  }
  uint32_t ob[B_INS];
#pragma unroll
  for (int i = 0; i < B_INS; ++i) {
    if constexpr (BKN) {
      // tile row = k (relative to the tile's first k), BN / 8 chunks per row; columns past N are
      // clamped onto the last full chunk (their results are never stored)
      constexpr int CPR = BN / 8;
      const int row = (i * NW + wid) * GB::RPI + lane / CPR;
      const int lc = (lane % CPR) ^ bkn_swz<BN>(row);
      ob[i] = 2u * (uint32_t)(row * (int)ldb + min(n0 + lc * 8, N - 8));
    } else {
      const int row = (i * NW + wid) * RPI + r_in;
      const int lc = DmaGeom<BKD>::swz(row, pc);
      ob[i] = 2u * (uint32_t)(min(n0 + row, N - 1) * (int)ldb + lc * 8);
    }
  }
  const uint32_t kb_step_b = 2u * (uint32_t)BKD * (uint32_t)ldb;  // B bytes per k-tile ([K, N] B)

  using Acc = typename MfmaAcc<MF>::type;
  Acc acc[NB][FM][FN];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < (int)(sizeof(Acc) / 4); ++e) acc[b][i][j][e] = 0.f;

  gemm_dma_ns_kloop<T, BM, BN, WM, WN, NB, BKD, NS, BKN, MF, SL>(acc, A, B0, B1, oa, ob, kb_step_b, K, wid, wm, wn,
                                                             lane, sS0, sS1, sS2, sS3);

  // 16x16 fragment: lane holds C[m0' + lane % 16][n0' + 4 (lane / 16) + 0..3]
  const int fr = lane & 15, fc = lane >> 4;
  if constexpr (EPI == kEpiStore && NB == 1 && kStage >= BM / 2 * BN && BN % 64 == 0) {
    if ((ldc & 1) != 0 || ((uintptr_t)C & 3) != 0) {  // uniform over the block
      store_tile_rows<T, BM, BN, NW, FM, FN>(C, ldc, M, N, m0, n0, wm * WTM, wn * WTN, acc[0], sS0, sS1);
      return;
    }
  }
  tile_epilogue<T, NB, EPI, true, FM, FN>(C, B1, ldc, M, N, m0 + wm * WTM + fr, n0 + wn * WTN + fc * 4, acc, ep);
}

// --------------------------------------------------------------------------------------------
// Host dispatch
// --------------------------------------------------------------------------------------------
struct TileCfg {
  int bm, bn;
};

// One tile row (M <= 64) reads B once, so what counts is how much of it is in flight. A 64x96 or 64x128
// tile has the CU to itself (four stages of LDS), two 64x64 ones share it and do not stop at each other's
// barriers. Whether the wider tiles of an [N, K] B are the faster ones (us, 64x64 / 64x128): they are on
// a grid well short of the CUs (1 x 20480 x 4096 38.1 / 33.1), or with many rows in the second round
// (64 x 50304 x 1024 27.0 / 24.1); not on a full one (1 x 32000 x 4096 49.8 / 57.8, 64 x 32000 x 4096 57.2 /
// 61.1) nor past two rounds (16 x 100000 x 2048 82 / 94). Of a [K, N] B, whose tile rows they make twice as
// long, they are the faster ones up to two rounds (16 x 50304 x 4096 83 / 74) and for deep K past them (64 x
// 100000 x 1024 57 / 51; but 64 x 100000 x 256 15.2 / 18.2). 128x192 tiles, two to a CU, waste more than half
// of each on such rows and lose the same way (1 x 200000 x 768 55 / 66).
static bool wide64_nt(int64_t M, int64_t N, int64_t K, int64_t waves) {
  if (waves == 1) return N <= 24576 || K < 2048;
  return waves == 2 && M > 32 && K >= 768;
}

// Pick the tile that keeps the 256 CUs busiest: fraction of CU-slots doing useful work over the
// launch, weighted by the per-tile efficiency of smaller tiles (more LDS and L2 traffic per flop).
// wide192: also consider 256x192 tiles (the LDS-DMA kernel with nn.Linear-layout B; 2048 x 6144,
// a fused QKV projection, is then exactly one tile per CU). small64: also consider 64x64 tiles
// (the same kernel, for grids that 128x128 tiles leave mostly idle) and 64x128 ones, and, with
// nn.Linear-layout B, 64x96 and 128x192 (whose weight is eff192, see kPairK).
// K: only for the rules of at most 64 rows.
static TileCfg pick_tile(int64_t M, int64_t N, int nb, bool wide192 = false, bool small64 = false,
                         int64_t batch = 1, double eff192 = 0.0, int64_t K = 0) {
  const TileCfg cands[] = {{256, 256}, {256, 128}, {128, 128}, {256, 192}, {64, 64}, {128, 192}, {64, 96}, {64, 128}};
  // relative per-flop throughput of the tiles (bf16, MI355X): 4096^3 on 256x256 1230 TF/s,
  // 2048x4096x4096 on 256x128 1084 TF/s, 2048x6144x4096 on 128x128 786 TF/s, on 256x192 1108 TF/s;
  // 64x64 weighted so that it wins only where 128x128 tiles fill under a third of the CUs (cold,
  // f16: 2048x768x768 16.4 -> 13.8 us, 2048x768x3072 41.7 -> 37.3 us, 1024^3 NN 17.3 -> 15.5 us,
  // 4096x768x768 unchanged at 15.1 us; with a weight of 0.5 it was also picked there and took
  // 16.3 us)
  // 64x96 and 64x128 lie between, by what a k-step of one tile on a CU takes (64x64 0.30 us, 64x96
  // 0.36, 64x128 0.44, 128x128 0.65, 128x192 0.80, 256x128 0.97), and win where they are what fills the
  // CUs (f16, NT, rotating operands, us, before / after): 2048x768x3072 28.1 / 21.9, 2048x768x768
  // 11.2 / 9.6, 512x2304x768 7.8 / 6.3 (64x96), 2048x1024x4096 34.1 / 28.7, 512x4096x4096 35.1 / 28.9
  // (64x128), 512x11008x4096 57.7 / 52.3 (128x192)
  const double eff[] = {1.0, 0.88, 0.64, 0.88, 0.35, eff192, 0.43, 0.47};
  const int cus = 256;
  TileCfg best = cands[2];
  double best_s = -1.0;
  for (int i = 0; i < 8; ++i) {
    const bool considered = i < 3 || (nb == 1 && (i == 3 ? wide192 : i == 5 ? eff192 > 0.0 : i == 6 ? small64 && wide192 : small64));
    if (!considered) continue;
    const int bn = cands[i].bn / (nb == 2 ? 2 : 1);
    const int64_t tiles = cdiv(M, cands[i].bm) * cdiv(N, bn) * batch;
    const int64_t waves = cdiv(tiles, cus);
    if (i == 5 && M <= 64 && waves > 1) continue;
    if (i >= 6 && M <= 64 && !(wide192 ? wide64_nt(M, N, K, waves) : waves <= 2 || (M > 8 && K >= 768))) continue;
    const double used = (double)tiles / (double)(waves * cus);
    // padding waste inside edge tiles
    const double pad = (double)(M * N) / (double)(cdiv(M, cands[i].bm) * cands[i].bm * cdiv(N, bn) * bn);
    const double s = used * pad * eff[i];
    if (s > best_s + 1e-9) {
      best_s = s;
      best = cands[i];
    }
  }
  return best;
}

template <typename T, bool BT, bool VEC, int BM, int BN, int WM, int WN, int NB, int EPI>
static void launch_gemm_cfg(const void* A, const void* B0, const void* B1, void* C, int M, int N,
                            int K, int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const EpiArgs& ep) {
  const int tiles_m = (int)cdiv(M, BM), tiles_n = (int)cdiv(N, BN);
  gemm_mfma<T, BT, VEC, BM, BN, WM, WN, NB, EPI><<<dim3(tiles_m * tiles_n, 1, ep.batch), WM * WN * kWave, 0, s>>>(
      (const uint16_t*)A, (const uint16_t*)B0, (const uint16_t*)B1, (uint16_t*)C, M, N, K, lda, ldb,
      ldc, tiles_m, tiles_n, ep);
}

// Waves along N of the 256x256 tile: 4 (8 waves of 128x64; measured faster than 4 waves of
// 128x128, one wave per SIMD with accumulators in AGPRs).
constexpr int kBigWN = 4;

template <typename T, bool BT, bool VEC, int NB, int EPI>
static void launch_gemm_tiled(const void* A, const void* B0, const void* B1, void* C, int M, int N,
                              int K, int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const EpiArgs& ep) {
  const TileCfg t = pick_tile(M, N, NB, false, false, ep.batch);
  if constexpr (NB == 1) {
    if (t.bm == 256 && t.bn == 256)
      launch_gemm_cfg<T, BT, VEC, 256, 256, 2, kBigWN, 1, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else if (t.bm == 256)
      launch_gemm_cfg<T, BT, VEC, 256, 128, 4, 2, 1, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else
      launch_gemm_cfg<T, BT, VEC, 128, 128, 2, 2, 1, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
  } else {
    if (t.bm == 256 && t.bn == 256)
      launch_gemm_cfg<T, BT, VEC, 256, 128, 2, 4, 2, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else if (t.bm == 256)
      launch_gemm_cfg<T, BT, VEC, 256, 64, 4, 2, 2, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else
      launch_gemm_cfg<T, BT, VEC, 128, 64, 2, 2, 2, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
  }
}

constexpr int kCUs = 256;  // MI355X compute units

// OCC: blocks that must fit on a CU together (it bounds the registers; LDS has to fit as well).
template <typename T, int BM, int BN, int WM, int WN, int NB, int EPI, int BKD, int NS, bool BKN, int OCC = 1, bool SL = false>
static void launch_dma_kernel(const void* A, const void* B0, const void* B1, void* C, int M, int N, int K,
                              int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles_n, hipStream_t s,
                              const EpiArgs& ep) {
  // MFMA shape 16x16x32 (32x32x16 fragments measured 4-10 % slower on every workload)
  constexpr int MF = 16;
  gemm_dma<T, BM, BN, WM, WN, NB, EPI, BKD, NS, BKN, MF, OCC, SL><<<dim3(tiles_m * tiles_n, ep.splits, ep.batch), WM * WN * kWave, 0, s>>>(
      (const uint16_t*)A, (const uint16_t*)B0, (const uint16_t*)B1, (uint16_t*)C, M, N, K, lda, ldb, ldc,
      tiles_m, tiles_n, ep);
}

// Pipeline plan per tile shape: stage bytes (BM + NB * BN) * BKD * 2 and the 160 KB of LDS fix
// how many stages fit.
// Waves along N of the 128x128 tile: 4 (8 waves of 64x32, two per SIMD). Measured, cold, 2048^3
// (256 tiles, one per CU): f16 NN 26.8 us against 36.5 us with 4 waves of 64x64 (stock hipBLASLt
// 32.0), bf16 NT 26.4 against 36.0 (28.9); three or four stages for the 4-wave tile reach
// 28.2-29.4 us. Shapes on other tiles are unchanged.
constexpr int kSmallWN = 4;

template <int BM, int BN, int NB, int NW>
struct DmaPlan {
  static constexpr int kStage64 = (BM + NB * BN) * 64 * 2;
  static constexpr int kFit64 = 163840 / kStage64;
  static constexpr bool kOk32 = BM % (16 * NW) == 0 && BN % (16 * NW) == 0;
  // Three 64-deep stages where they fit beside 8 waves, else two. Measured (bf16, NT):
  // 2048x4096x4096 on 256x128 tiles 83.5 us two-stage -> 63.4 us three-stage; 4096^3 on 256x256
  // 107.4 us two-stage (four 32-deep stages: 121.2 us, the doubled barrier count outweighs the
  // deeper queue). The tiles of 64 rows (4 waves, 16 - 24 KB stages, picked for grids that larger
  // tiles leave mostly idle) wait on transfer latency, not MFMAs: four stages keep three tiles in
  // flight (cold, f16, 64x64: 1024^3 15.5 -> 10.8 us, 2048x768x3072 37.0 -> 29.8 us, 2048x1024x1024
  // 16.6 -> 14.6 us; six or eight stages, or four on 128x128 tiles, gained nothing).
  static constexpr int BKD = 64;
  static constexpr int NS = BM == 64 ? 4 : (kFit64 >= 3 && NW == 8) ? 3 : 2;
};

template <typename T, int BM, int BN, int WM, int WN, int NB, int EPI, bool BKN>
static void launch_dma_cfg(const void* A, const void* B0, const void* B1, void* C, int M, int N, int K,
                           int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const EpiArgs& ep) {
  const int tiles_m = (int)cdiv(M, BM), tiles_n = (int)cdiv(N, BN);
  using P = DmaPlan<BM, BN, NB, WM * WN>;
  // Four 32-deep stages when the grid fills at most half the CUs (each block's own DMA latency is
  // then exposed; measured 2048x1024x4096: 50.9 us against 59.0 us two-stage). With more tiles the
  // 64-deep pair is faster per tile (2048x6144x4096 on 192 tiles of 256x256: 109.9 us against
  // 127.5 us).
  // 64-row tiles keep their four 64-deep stages there (f16: 128x768x768 7.3 us 32-deep, 6.3 64-deep;
  // 512x768x3072 23.1, 17.4) unless K is so short that most of what they fetch is past it (12x128x64 nn 2.95,
  // 3.15; 112x1344x64 nn 3.36, 3.59).
  constexpr bool kOk32 = P::kOk32;
  if (kOk32 && (BM > 64 || K <= 128) && 2 * tiles_m * tiles_n * ep.splits * ep.batch <= kCUs) {
    if constexpr (kOk32)
      launch_dma_kernel<T, BM, BN, WM, WN, NB, EPI, 32, 4, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, tiles_m,
                                                                tiles_n, s, ep);
    return;
  }
  launch_dma_kernel<T, BM, BN, WM, WN, NB, EPI, P::BKD, P::NS, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, tiles_m,
                                                                    tiles_n, s, ep);
}

// Largest K for which 128x192 tiles are considered. A product of few k-steps spends about as long in
// each tile's first loads and in its epilogue (bias, GELU, residual, stores) as in its MFMAs, and the
// larger tiles have the CU to themselves, so nothing runs meanwhile. Two blocks of 8 waves and two
// 40 KB stages share a CU, and one multiplies while the other stores. Measured (f16, NT, rotating
// operands, us, before / after): 2048x3072x768 + GELU 25.0 / 21.0, 8192x3072x768 + GELU 75.8 / 61.4,
// 2048x2304x768 15.2 / 13.8, 8192x2304x768 42.6 / 36.0, 8192x768x768 + residual 20.4 / 18.7,
// 1000x5000x1024 17.0 / 16.2. A long K hides both ends and wants the larger tile's fewer LDS reads
// per flop (8192x768x3072 53.8 / 55.0, 4096x11008x4096 317 / 350): there a 128x192 tile has the CU and
// three stages to itself and is picked where it is what fills the chip.
// Their weight among pick_tile's lies where they are level with the others: 256x192 tiles of which
// every CU gets one (4096x3072x768 + bias 26.1 us as pairs, 24.1; 4096x2304x768 + bias 23.4, 22.5)
// stay, except under the GELU, whose 50 instructions an output the pair hides (4096x3072x768 + GELU
// 33.2, 34.9); 1024x2304x768 stays on 128x128 tiles (13.3, 9.2).
constexpr int kPairK = 1024;
template <int EPI>
constexpr double kPairEff = EPI == kEpiBiasGelu ? 0.9 : 0.86;
constexpr double kLongEff192 = 0.77;

template <typename T, int NB, int EPI, bool BKN>
static void launch_gemm_dma(const void* A, const void* B0, const void* B1, void* C, int M, int N, int K,
                            int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const EpiArgs& ep) {
  // 256x192 needs [N, K] B: a [K, N] B tile row of 192 elements does not split into 1 KB transfers
  constexpr bool kPair = NB == 1 && !BKN && EPI != kEpiPartial;
  const TileCfg t = pick_tile(M, N, NB, !BKN, EPI != kEpiPartial, ep.batch, !kPair ? 0.0 : K <= kPairK ? kPairEff<EPI> : kLongEff192, K);
  if constexpr (NB == 1) {
    if constexpr (kPair) {
      if (t.bm == 128 && t.bn == 192) {
        const int tm = (int)cdiv(M, 128), tn = (int)cdiv(N, 192);
        if (K <= kPairK) launch_dma_kernel<T, 128, 192, 2, 4, 1, EPI, 64, 2, false, 2>(A, B0, B1, C, M, N, K, lda, ldb, ldc, tm, tn, s, ep);
        else launch_dma_kernel<T, 128, 192, 2, 4, 1, EPI, 64, 3, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, tm, tn, s, ep);
        return;
      }
      if (t.bm == 64 && t.bn == 96) {
        launch_dma_cfg<T, 64, 96, 2, 2, 1, EPI, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
        return;
      }
    }
    if constexpr (EPI != kEpiPartial) {
      if (t.bm == 64 && t.bn == 128) {
        launch_dma_cfg<T, 64, 128, 2, 2, 1, EPI, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
        return;
      }
    }
    if constexpr (!BKN) {
      if (t.bm == 256 && t.bn == 192) {
        launch_dma_cfg<T, 256, 192, 2, 4, 1, EPI, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
        return;
      }
    }
    if (t.bm == 64) {
      launch_dma_cfg<T, 64, 64, 2, 2, 1, EPI, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
      return;
    }
    if (t.bm == 256 && t.bn == 256)
      launch_dma_cfg<T, 256, 256, 2, kBigWN, 1, EPI, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else if (t.bm == 256) launch_dma_cfg<T, 256, 128, 4, 2, 1, EPI, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else launch_dma_cfg<T, 128, 128, 2, kSmallWN, 1, EPI, BKN>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
  } else {
    static_assert(!BKN, "gate/up weights are [H, D]");
    if (t.bm == 256 && t.bn == 256)
      launch_dma_cfg<T, 256, 128, 2, kBigWN, 2, EPI, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else if (t.bm == 256) launch_dma_cfg<T, 256, 64, 4, 2, 2, EPI, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
    else launch_dma_cfg<T, 128, 64, 2, 2, 2, EPI, false>(A, B0, B1, C, M, N, K, lda, ldb, ldc, s, ep);
  }
}

// A batch of products that each take gemm_small, summed in its order by tiles: past 512 blocks of 32 x 32 the
// tiles, which share their operands' loads, are the faster form (us, a block's 16 waves / four slices a wave / these:
// f16 nt 64 x 64 x 512, 128 items 22 / 10 / 8.5, 512 items 76 / 27 / 16; 64 x 1024 x 1024, 4 items 15 / 8 / 13, 128 items 425 /
// 137 / 76; nn 32 x 3000 x 1000, 8 items 33 / 38 / 24). dma: the LDS-DMA kernel reads them; vec: 16-byte loads do.
template <typename T>
static int launch_gemm_slices(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb,
                              int64_t ldc, bool bt, bool dma, bool vec, hipStream_t s, const EpiArgs& ep) {
  const int tm = (int)cdiv(M, 64), tn = (int)cdiv(N, 64);
  if (!dma) {
#define AK_SL(BT, VEC, SL)                                                                                       \
  gemm_mfma<T, BT, VEC, 64, 64, 2, 2, 1, kEpiStore, SL><<<dim3(tm * tn, 1, ep.batch), 4 * kWave, 0, s>>>(        \
      (const uint16_t*)A, (const uint16_t*)B, nullptr, (uint16_t*)C, M, N, K, lda, ldb, ldc, tm, tn, ep)
#define AK_SLV(BT, SL)              \
  {                                 \
    if (vec) AK_SL(BT, true, SL);   \
    else AK_SL(BT, false, SL);      \
  }
    if (small_k64(M, N, bt)) {
      if (bt) AK_SLV(true, 64) else AK_SLV(false, 64)
    } else {
      if (bt) AK_SLV(true, 32) else AK_SLV(false, 32)
    }
#undef AK_SLV
#undef AK_SL
    return record_launch();
  }
#define AK_SL(BKD, BKN) \
  launch_dma_kernel<T, 64, 64, 2, 2, 1, kEpiStore, BKD, 4, BKN, 2, true>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, tm, tn, s, ep)
  if (small_k64(M, N, bt)) {
    if (bt) AK_SL(64, false);
    else AK_SL(64, true);
  } else {
    if (bt) AK_SL(32, false);
    else AK_SL(32, true);
  }
#undef AK_SL
  return record_launch();
}

// Products of at most kSmallM rows on operands the LDS-DMA kernel can read: whether gemm_small is the
// faster one. Measured (bf16, three rotating operand sets, us, LDS-DMA unsplit / gemm_small, M = 1, 16,
// 32, 64; "nt" is an [N, K] B):
//   nt N 2304 K 768    5.6 5.9 5.8 5.9 / 4.3 4.8 5.2 6.4     nt N 4096 K 4096   19.2 19.3 19.7 20.6 / 9.3 11.2 14.6 18.5
//   nt N 4096 K 11008  56 58 60 75 / 18 26 35 45             nt N 8192 K 4096   20.0 20.0 20.5 21.5 / 19.4 21.7 26.0 26.3
//   nn N 768 K 2048    10.0 10.1 10.2 10.4 / 5.4 6.1 6.2 6.5 nn N 4096 K 768    5.5 5.7 5.8 5.9 / 5.4 5.7 6.7 6.8
//   nn N 4096 K 4096   18.9 19.1 19.2 20.6 / 15.3 16.0 18.8 18.7
// Past N = 4096 the LDS-DMA kernel's tiles fill enough of the chip, and below K = 512 both are launches.
// Gate/up (LDS-DMA / gemm_small, M = 1, 16, 32, 64): 4096 -> 11008 65 65 66 65 / 50 55 61 81, 768 -> 2048
// 10.5 12.5 10.6 10.8 / 5.0 5.4 6.8 6.6, 192 -> 11648 7.3 7.3 7.5 8.1 / 7.7 8.1 6.9 9.7.
static bool small_rows_win(int64_t M, int64_t N, int64_t K, bool bt, int nb) {
  if (nb == 2) return N <= 4096 || (M <= 32 && K >= 512);
  if (N > 4096 || K < 512) return false;
  if (bt) return M <= 32 || N <= 1024 || K >= 2048;
  return N <= 2560 || K >= 2048;
}

// Shapes and row strides the LDS-DMA path serves (aligned operands provided): K a multiple of 64, 16-byte
// chunks, 32-bit element offsets.
static bool dma_shape(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, bool bt) {
  return K > 0 && K % kBK == 0 && lda % 8 == 0 && ldb % 8 == 0 && (bt || N % 8 == 0) && M * lda < INT_MAX &&
         (bt ? N : K) * ldb < INT_MAX;
}

// The period of a batch's kernel choice. A product of at most kSmallM rows that small_rows_win leaves to
// the LDS-DMA kernel takes gemm_small where its operands are off 16 bytes, and the two sum in different
// orders. Every item of a batch has to equal its 2-D product, so where the batch strides move items on
// and off 16 bytes, the aligned ones (z, z + p, ... for one z) are a launch of their own.
static int64_t batch_period(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t stride_a,
                            int64_t stride_b, bool bt) {
  if (M > kSmallM || N > small_max_n(1) || !dma_shape(M, N, K, lda, ldb, bt) || small_rows_win(M, N, K, bt, 1)) return 1;
  int64_t p = 1;
  while ((p * stride_a) % 8 != 0 || (p * stride_b) % 8 != 0) p *= 2;
  return p;
}

template <typename T, int NB, int EPI>
static int launch_gemm16(const void* A, const void* B0, const void* B1, void* C, int64_t M,
                         int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, bool bt,
                         hipStream_t s, const EpiArgs& ep = EpiArgs{}) {
  // vec: A and B load as 16-byte k-chunks. C's alignment does not matter, nor does that of a bias or a
  // residual (B1 of one product): the epilogue checks each 8-byte access. They must not choose the kernel
  // either, whose order of the sums an epilogue shares with the plain product.
  bool vec = K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && (bt || N % 8 == 0) && host_aligned16(A) && host_aligned16(B0) &&
             (NB == 1 || host_aligned16(B1)) && ep.skip < 0;
  const int m = (int)M, n = (int)N, k = (int)K;
  const bool dma = vec && dma_shape(M, N, K, lda, ldb, bt);
  // Few rows: always for operands that path cannot read, by shape for those it can.
  if (M <= kSmallM && N <= small_max_n(NB) && K > 0 && (bt || NB == 1) && (!dma || small_rows_win(M, N, K, bt, NB))) {
    if constexpr (NB == 1 && EPI == kEpiStore) {
      if (ep.batch > 1 && M > 16 && N <= 4096 && K <= (1 << 30) && cdiv(M, 32) * cdiv(N, 32) * ep.batch >= 512) {
        const bool vz = vec && ep.batch_a % 8 == 0 && ep.batch_b % 8 == 0;
        return launch_gemm_slices<T>(A, B0, C, m, n, k, lda, ldb, ldc, bt, dma && vz, vz, s, ep);
      }
    }
    return launch_gemm_small<T, NB, EPI>(A, B0, B1, C, M, N, K, lda, ldb, ldc, bt, s, ep);
  }
  vec = vec && ep.batch_a % 8 == 0 && ep.batch_b % 8 == 0;
  if (bt && dma && vec) {
    launch_gemm_dma<T, NB, EPI, false>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
    return record_launch();
  }
  // [K, N] B (torch.matmul's layout) on the same pipeline, fragments read through LDS transposes
  if constexpr (NB == 1) {
    if (!bt && dma && vec) {
      launch_gemm_dma<T, 1, EPI, true>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
      return record_launch();
    }
  }
  if (bt) {
    if (vec) launch_gemm_tiled<T, true, true, NB, EPI>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
    else launch_gemm_tiled<T, true, false, NB, EPI>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
  } else {
    if constexpr (NB == 1) {
      if (vec) launch_gemm_tiled<T, false, true, 1, EPI>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
      else launch_gemm_tiled<T, false, false, 1, EPI>(A, B0, B1, C, m, n, k, lda, ldb, ldc, s, ep);
    } else {
      return AK_EINVAL;
    }
  }
  return record_launch();
}

// ---------------------------------------------------------------------------------------------
// Split-K for grids that leave most CUs idle (few output tiles, long K): slice z of the K range runs
// as grid row z of the LDS-DMA kernel and stores fp32 partial tiles to the caller's workspace
// [splits][M][N]; splitk_reduce then adds the slices in order z = 0, 1, ... and rounds once, so the
// result is deterministic and keeps "fp32 accumulation, one output rounding".
// ---------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce(const float* __restrict__ ws, uint16_t* __restrict__ C, int M,
                                                     int N, int64_t ldc, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one 4-column group per thread
  const int groups_per_row = N / 4;
  if (i >= (int64_t)M * groups_per_row) return;
  const int m = (int)(i / groups_per_row), n = (int)(i % groups_per_row) * 4;
  const int64_t plane = (int64_t)M * N;
  const float* p = ws + (int64_t)m * N + n;
  f32x4 acc = *reinterpret_cast<const f32x4*>(p);
  for (int z = 1; z < splits; ++z) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(p + z * plane);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += v[e];
  }
  u32x2 o;
  o[0] = (uint32_t)T::from_f(acc[0]) | ((uint32_t)T::from_f(acc[1]) << 16);
  o[1] = (uint32_t)T::from_f(acc[2]) | ((uint32_t)T::from_f(acc[3]) << 16);
  *reinterpret_cast<u32x2*>(C + (int64_t)m * ldc + n) = o;
}

// K slices for a plain f16 / bf16 GEMM on the LDS-DMA path, 1 when splitting does not pay: the
// chosen tiling must fill at most half the CUs, each slice keeps at least 1024 of K (sixteen
// 64-deep tiles) and a multiple of 64, and slices stop doubling once tiles x slices would pass the
// CU count.
static int splitk_slices(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, bool bt) {
  if (M <= kSmallM) {
    // gemm_small splits K inside its blocks, and is the faster one while its few columns are read by
    // 16 rows or fewer or the matrix is small (us, split LDS-DMA / gemm_small: nt 16 x 4096 x 4096 14.2 /
    // 11.2, nt 64 x 768 x 11008 26.8 / 22.9, nn 16 x 4096 x 2048 12.9 / 9.8; but nt 32 x 4096 x 11008
    // 31.8 / 35.3, nn 16 x 4096 x 4096 14.4 / 16.0)
    if (bt ? N <= 1024 || (N <= 4096 && M <= 16) : (N <= 768 && K <= 8192) || (N <= 4096 && K < 4096)) return 1;
    // more than 128 tiles of 64 columns fill the chip unsplit (nt 16 x 11008 x 4096: 18.2 us against 21.6
    // in two slices of 128 x 128 tiles; 128 tiles, N = 8192: 20.0 against 16.1); a deep [K, N] B still
    // gains (nn 32 x 11008 x 11008: 55.1 us split, 59.4 unsplit)
    if (cdiv(N, 64) > 128 && (bt || K <= 8192)) return 1;
  }
  if (M <= 0 || N <= 0 || K <= 0 || N % 4 != 0 || ldc % 4 != 0 || lda % 8 != 0 || ldb % 8 != 0) return 1;
  if (M * lda >= INT_MAX || (bt ? N : K) * ldb >= INT_MAX || M * N * 8 >= INT_MAX) return 1;
  // [K, N] B runs the LDS-DMA kernel only with N a multiple of 8 (its 16-byte column chunks), the
  // same rule as the unsplit path
  if (!bt && N % 8 != 0) return 1;
  const TileCfg t = pick_tile(M, N, 1, !bt);
  const int64_t tiles = cdiv(M, t.bm) * cdiv(N, t.bn);
  if (2 * tiles > kCUs) return 1;
  int s = 1;
  // Slices stay at least 1024 deep: shorter ones lose more to the pipeline fill and the fp32
  // partial round trip than the extra CUs win (1024^3 f16: 11.9 us unsplit, 18.0 us in 4 slices;
  // 1024x1024x4096: 32.5 us unsplit, 22.8 us in 4 slices).
  while (s < 8 && tiles * s * 2 <= kCUs && K % (64 * s * 2) == 0 && K / (s * 2) >= 1024) s *= 2;
  return s;
}

template <typename T>
static int launch_gemm16_splitk(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                                int64_t lda, int64_t ldb, int64_t ldc, bool bt, int splits, float* ws,
                                hipStream_t s) {
  EpiArgs ep;
  ep.splits = splits;
  const int64_t ks = K / splits;
  ep.split_a = ks;
  ep.split_b = bt ? ks : ks * ldb;
  ep.split_c = M * N;
  // partial tiles: the workspace is the output, row stride N
  if (bt) launch_gemm_dma<T, 1, kEpiPartial, false>(A, B, nullptr, ws, (int)M, (int)N, (int)ks, lda, ldb, N, s, ep);
  else launch_gemm_dma<T, 1, kEpiPartial, true>(A, B, nullptr, ws, (int)M, (int)N, (int)ks, lda, ldb, N, s, ep);
  const int64_t groups = M * (N / 4);
  splitk_reduce<T><<<(unsigned)cdiv(groups, 256), 256, 0, s>>>(ws, (uint16_t*)C, (int)M, (int)N, ldc, splits);
  return record_launch();
}

}  // namespace ak

using namespace ak;

extern "C" int ak_gemm(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N,
                       int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int b_trans,
                       hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  const bool bt = b_trans != 0;
  switch (dtype) {
    case AK_F32: return launch_gemm32(A, B, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_F16: return launch_gemm16<TF16, 1, kEpiStore>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiStore>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, bt, stream);
    default: return AK_EINVAL;
  }
}

extern "C" int ak_gemm_batched(int dtype, const void* A, const void* B, void* C, int64_t batch, int64_t M,
                               int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t stride_a,
                               int64_t stride_b, int64_t stride_c, int b_trans, hipStream_t stream) {
  if (batch < 0 || M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (batch == 0 || M == 0 || N == 0) return AK_OK;
  if (!A || !B || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N) || stride_a < 0 || stride_b < 0) return AK_EINVAL;
  // the batch items of C must not overlap (each is written once, in parallel)
  if (batch > 1 && stride_c < (M - 1) * ldc + N) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  const bool bt = b_trans != 0;
  const int esz = dtype == AK_F32 ? 4 : 2;
  const int64_t period = dtype == AK_F32 ? 1 : batch_period(M, N, K, lda, ldb, stride_a, stride_b, bt);
  // the items both of whose operands are aligned: one of the first `period`, and every period-th after it
  int64_t own = -1;
  if (period > 1)
    for (int64_t z = 0; z < period && own < 0; ++z)
      if (host_aligned16((const char*)A + z * stride_a * esz) && host_aligned16((const char*)B + z * stride_b * esz)) own = z;
  // items first, first + step, ...; skip: leave the aligned ones out
  auto launch = [&](int64_t first, int64_t step, bool skip) -> int {
    const int64_t sa = stride_a * step, sb = stride_b * step, sc = stride_c * step;
    // grid z holds at most 65535 items: larger batches run in chunks
    constexpr int64_t kMaxZ = 65535;
    const int64_t items = cdiv(batch - first, step);
    for (int64_t z0 = 0; z0 < items; z0 += kMaxZ) {
      const int64_t nz = items - z0 < kMaxZ ? items - z0 : kMaxZ, z = first + z0 * step;
      const char* a = (const char*)A + z * stride_a * esz;
      const char* b = (const char*)B + z * stride_b * esz;
      char* c = (char*)C + z * stride_c * esz;
      int st = AK_OK;
      if (dtype == AK_F32) {
        st = launch_gemm32(a, b, c, M, N, K, lda, ldb, ldc, bt, stream, (int)nz, sa, sb, sc);
      } else {
        EpiArgs ep;
        ep.batch = (int)nz;
        ep.batch_a = sa;
        ep.batch_b = sb;
        ep.batch_c = sc;
        if (skip) {
          ep.skip = (int)((own + period - z0 % period) % period);
          ep.skip_period = (int)period;
        }
        if (dtype == AK_F16) st = launch_gemm16<TF16, 1, kEpiStore>(a, b, nullptr, c, M, N, K, lda, ldb, ldc, bt, stream, ep);
        else if (dtype == AK_BF16) st = launch_gemm16<TBF16, 1, kEpiStore>(a, b, nullptr, c, M, N, K, lda, ldb, ldc, bt, stream, ep);
        else return AK_EINVAL;
      }
      if (st != AK_OK) return st;
    }
    return AK_OK;
  };
  if (own < 0 || own >= batch) return launch(0, 1, false);
  const int st = launch(own, period, false);
  return st == AK_OK && batch > 1 ? launch(0, 1, true) : st;
}

extern "C" int64_t ak_gemm_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                           int64_t ldc, int b_trans) {
  if (dtype != AK_F16 && dtype != AK_BF16) return 0;
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return 0;
  const int sl = splitk_slices(M, N, K, lda, ldb, ldc, b_trans != 0);
  return sl > 1 ? (int64_t)sl * M * N * (int64_t)sizeof(float) : 0;
}

extern "C" int ak_gemm_ws(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                          int64_t lda, int64_t ldb, int64_t ldc, int b_trans, void* workspace,
                          int64_t workspace_bytes, hipStream_t stream) {
  const int64_t need = ak_gemm_workspace_bytes(dtype, M, N, K, lda, ldb, ldc, b_trans);
  const bool aligned = host_aligned16(A) && host_aligned16(B) && (((uintptr_t)C) & 7u) == 0 &&
                       host_aligned16(workspace);
  if (need == 0 || !workspace || workspace_bytes < need || !aligned || lda < K || ldc < N ||
      ldb < (b_trans ? K : N))
    return ak_gemm(dtype, A, B, C, M, N, K, lda, ldb, ldc, b_trans, stream);
  const int sl = (int)(need / (M * N * (int64_t)sizeof(float)));
  if (dtype == AK_F16)
    return launch_gemm16_splitk<TF16>(A, B, C, M, N, K, lda, ldb, ldc, b_trans != 0, sl, (float*)workspace, stream);
  return launch_gemm16_splitk<TBF16>(A, B, C, M, N, K, lda, ldb, ldc, b_trans != 0, sl, (float*)workspace, stream);
}

extern "C" int ak_gemm_residual(int dtype, const void* A, const void* B, const void* R, void* C, int64_t M,
                                int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int b_trans,
                                hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !R || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  // R is read and C written element by element in one pass: they must not overlap
  const uintptr_t r0 = (uintptr_t)R, c0 = (uintptr_t)C;
  const uintptr_t span = (uintptr_t)(((M - 1) * ldc + N) * 2);
  if (r0 < c0 + span && c0 < r0 + span) return AK_EINVAL;
  const bool bt = b_trans != 0;
  switch (dtype) {
    case AK_F16: return launch_gemm16<TF16, 1, kEpiResidual>(A, B, R, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiResidual>(A, B, R, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_F32: return AK_EUNSUPPORTED;
    default: return AK_EINVAL;
  }
}

extern "C" int ak_gemm_bias(int dtype, const void* A, const void* B, const void* bias, void* C, int64_t M,
                            int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int b_trans,
                            hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !bias || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  const bool bt = b_trans != 0;
  switch (dtype) {
    case AK_F16: return launch_gemm16<TF16, 1, kEpiBias>(A, B, bias, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiBias>(A, B, bias, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_F32: return AK_EUNSUPPORTED;
    default: return AK_EINVAL;
  }
}

extern "C" int ak_gemm_bias_gelu(int dtype, const void* A, const void* B, const void* bias, void* C, int64_t M,
                                 int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int b_trans,
                                 hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !bias || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  const bool bt = b_trans != 0;
  switch (dtype) {
    case AK_F16: return launch_gemm16<TF16, 1, kEpiBiasGelu>(A, B, bias, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiBiasGelu>(A, B, bias, C, M, N, K, lda, ldb, ldc, bt, stream);
    case AK_F32: return AK_EUNSUPPORTED;
    default: return AK_EINVAL;
  }
}

extern "C" int ak_gemm_bias_residual(int dtype, const void* A, const void* B, const void* bias, const void* R,
                                     void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                     int64_t ldc, int b_trans, hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !bias || !R || !C) return AK_EINVAL;
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  // R is read and C written element by element in one pass: they must not overlap
  const uintptr_t r0 = (uintptr_t)R, c0 = (uintptr_t)C;
  const uintptr_t span = (uintptr_t)(((M - 1) * ldc + N) * 2);
  if (r0 < c0 + span && c0 < r0 + span) return AK_EINVAL;
  const bool bt = b_trans != 0;
  EpiArgs ep;
  ep.bias = (const uint16_t*)bias;
  switch (dtype) {
    case AK_F16: return launch_gemm16<TF16, 1, kEpiBiasResidual>(A, B, R, C, M, N, K, lda, ldb, ldc, bt, stream, ep);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiBiasResidual>(A, B, R, C, M, N, K, lda, ldb, ldc, bt, stream, ep);
    case AK_F32: return AK_EUNSUPPORTED;
    default: return AK_EINVAL;
  }
}

extern "C" int ak_gemm_rope(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                            int64_t lda, int64_t ldb, int64_t ldc, int b_trans, const float* cos_t,
                            const float* sin_t, int64_t seq_len, int64_t head_dim, int64_t rot_cols,
                            hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX) return AK_EINVAL;
  if (head_dim <= 0 || head_dim % 4 != 0 || head_dim > INT_MAX) return AK_EINVAL;
  if (rot_cols < 0 || rot_cols > N || rot_cols % head_dim != 0) return AK_EINVAL;
  if (seq_len <= 0 || seq_len > INT_MAX) return AK_EINVAL;
  if (M == 0 || N == 0) return AK_OK;
  if (!A || !B || !C || (rot_cols > 0 && (!cos_t || !sin_t))) return AK_EINVAL;
  if ((((uintptr_t)cos_t) | ((uintptr_t)sin_t)) & 7u) return AK_EINVAL;  // pairs load as 8 bytes
  if (lda < K || ldc < N || ldb < (b_trans ? K : N)) return AK_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > INT_MAX) return AK_EINVAL;
  EpiArgs ep;
  ep.cos = cos_t;
  ep.sin = sin_t;
  ep.head_dim = (int)head_dim;
  ep.rot_cols = (int)rot_cols;
  ep.seq_len = (int)seq_len;
  const bool bt = b_trans != 0;
  switch (dtype) {
    case AK_F16: return launch_gemm16<TF16, 1, kEpiRope>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, bt, stream, ep);
    case AK_BF16: return launch_gemm16<TBF16, 1, kEpiRope>(A, B, nullptr, C, M, N, K, lda, ldb, ldc, bt, stream, ep);
    case AK_F32: return AK_EUNSUPPORTED;
    default: return AK_EINVAL;
  }
}

extern "C" int ak_mlp_gate_up(int dtype, const void* x, const void* w_gate, const void* w_up, void* h,
                              int64_t M, int64_t H, int64_t D, int activation, hipStream_t stream) {
  if (M < 0 || H < 0 || D < 0 || M > INT_MAX || H > INT_MAX || D > INT_MAX) return AK_EINVAL;
  if (M == 0 || H == 0) return AK_OK;
  if (!x || !w_gate || !w_up || !h) return AK_EINVAL;
  int epi;
  switch (activation) {
    case AK_ACT_SILU: epi = kEpiSilu; break;
    case AK_ACT_GELU: epi = kEpiGelu; break;
    case AK_ACT_RELU2: epi = kEpiRelu2; break;
    case AK_ACT_NONE: epi = kEpiNone; break;
    default: return AK_EINVAL;
  }
  if (dtype == AK_F32) return launch_gate_up32(x, w_gate, w_up, h, M, H, D, epi, stream);
#define AK_GU(TT)                                                                                          \
  switch (epi) {                                                                                           \
    case kEpiSilu: return launch_gemm16<TT, 2, kEpiSilu>(x, w_gate, w_up, h, M, H, D, D, D, H, true, stream);   \
    case kEpiGelu: return launch_gemm16<TT, 2, kEpiGelu>(x, w_gate, w_up, h, M, H, D, D, D, H, true, stream);   \
    case kEpiRelu2: return launch_gemm16<TT, 2, kEpiRelu2>(x, w_gate, w_up, h, M, H, D, D, D, H, true, stream); \
    default: return launch_gemm16<TT, 2, kEpiNone>(x, w_gate, w_up, h, M, H, D, D, D, H, true, stream);         \
  }
  if (dtype == AK_F16) { AK_GU(TF16) }
  if (dtype == AK_BF16) { AK_GU(TBF16) }
#undef AK_GU
  return AK_EINVAL;
}

// gemm_small.hip -- products with at most 64 rows of A (a decode step's tokens): f16 / bf16 / fp32, both
// B layouts, every epilogue of the GEMM entry points, and the SwiGLU gate/up.
//
// What bounds it: reading B (the weights) once from HBM. The tile kernels of gemm.hip give such a
// product few blocks, each walking K through LDS stages behind barriers; here
//   * a block owns 16 CF columns ([N, K] B) or 64 columns ([K, N] B) and all rows, and its WV waves
//     split K: wave w takes the groups of U k-steps w, w + WV, ... (neighbouring waves read
//     neighbouring parts of the same B rows), with the next group's loads in flight while it
//     multiplies. No LDS and no barrier until the end;
//   * operands go from global memory to the MFMA registers: a lane's 16 bytes of an A row or a
//     [N, K] B row are one operand. Of a [K, N] B a lane loads 4 columns of each k it needs (one row
//     of 64 columns per 16 lanes): fragment e holds columns 4 i + e, 16-bit k pairs are put together
//     with v_perm_b32, and fp32 needs no regrouping. Loads take any alignment, so no operand is
//     repacked; the K tail and a ragged right edge load elements, zeros past the end;
//   * the waves' partial sums are added through LDS in a fixed tree (deterministic), for fp32 with
//     their compensations (two-sum), so splitting K costs no accuracy. One wave per 16 rows then runs
//     the epilogue.
// Measured (us, before / now; three rotating operand sets): bf16 nt 1 x 4096 x 4096 13.9 / 9.4, 16 x 4096 x
// 11008 30 / 26, nn 29 x 3702 x 10112 (repacked before) 237 / 64, nn 10 x 1536 x 246 28 / 12; gate/up
// 16 x 4096 -> 11008 65 / 55; f32 nt 16 x 11008 x 4096 563 / 57, nn 28 x 553 x 6656 940 / 53.
// The slices (WV, or WV LV) and U, which fix the order of the sums, depend on M, N, B's layout and NB only, so that a batched
// product equals its items, and an epilogue equals the separate op, bit for bit. Which products come here
// also depends on the alignment of A and B (launch_gemm16), which a product and its epilogue forms share;
// ak_gemm_batched launches the aligned items of a batch apart where that decides (batch_period), and large
// batches run in the same order on other kernels (launch_gemm_small, launch_gemm_slices).
#include <limits.h>

#include "gemm_common.h"

namespace ak {

// Vector accesses at element alignment: 16 bytes of a row, and VN columns of one k.
template <typename S, int VN>
struct SmallVec {
  typedef u32x4 V16 __attribute__((aligned(2)));
  typedef uint32_t R __attribute__((ext_vector_type(VN * (int)sizeof(S) / 4)));
  struct __attribute__((packed, aligned(2))) VR {
    R v;
  };
};

// A compensated sum's correction for the next step. Of a finite total it is at most 2^104 (half a unit in
// the last place of the largest total, and the rounding of t - s). Once the total is infinite it is
// NaN or an infinity of the other sign, and the next step would turn the total into NaN; bounded
// (v_med3_f32 takes a NaN to a finite bound), it leaves an infinite total as it is, as a plain sum does.
// One VALU operation more per element and 16 of k, hidden behind the loads.
__device__ __forceinline__ float kahan_bound(float y) { return __builtin_amdgcn_fmed3f(y, -0x1p104f, 0x1p104f); }

// the first `valid` elements of p (16 bytes, or VN columns), zeros after
template <typename S>
__device__ __forceinline__ u32x4 small_load_k(const S* p, int valid) {
  constexpr int KV = 16 / (int)sizeof(S);
  u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < KV; ++e) {
    if constexpr (sizeof(S) == 2) {
      const uint32_t h = e < valid ? p[e] : 0u;
      v[e >> 1] |= h << ((e & 1) * 16);
    } else {
      v[e] = e < valid ? __builtin_bit_cast(uint32_t, p[e]) : 0u;
    }
  }
  return v;
}
template <typename S, int VN>
__device__ __forceinline__ typename SmallVec<S, VN>::R small_load_n(const S* p, int valid) {
  typename SmallVec<S, VN>::R v;
#pragma unroll
  for (int e = 0; e < VN; ++e) {
    if constexpr (sizeof(S) == 2) {
      const uint32_t h = e < valid ? p[e] : 0u;
      v[e >> 1] = (e & 1) ? v[e >> 1] | (h << 16) : h;
    } else {
      v[e] = e < valid ? __builtin_bit_cast(uint32_t, p[e]) : 0u;
    }
  }
  return v;
}

// Waves per SIMD the registers allow without spills.
constexpr int small_occupancy(int wv, int lv, int mf, bool bt, bool f32) {
  return lv > 1 ? 2 : wv == 16 || (bt && (mf == 1 || (mf == 4 && !f32))) ? 4 : bt && mf == 2 ? 3 : 2;
}

// LV: the K slices of a wave. With LV = 1 wave w adds slice w; with more it adds slices w, w + WV, ... one
// after another and puts them together in registers in the order the tree over WV LV waves would.
template <typename T, bool BT, int NB, int EPI, int MF, int CF, int WV, int LV, int U>
__global__ __launch_bounds__(WV* kWave, small_occupancy(WV, LV, MF, BT, sizeof(typename T::S) == 4)) void gemm_small(
    const typename T::S* __restrict__ A, const typename T::S* __restrict__ B0, const typename T::S* __restrict__ B1,
    typename T::S* __restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, EpiArgs ep) {
  using S = typename T::S;
  constexpr int VN = BT ? 4 : CF;          // [K, N] B: columns per lane
  using SV = SmallVec<S, VN>;
  constexpr bool F32 = sizeof(S) == 4;
  constexpr int KV = 16 / (int)sizeof(S);  // k per lane and step
  constexpr int KS = 4 * KV;               // k per step: 32 (one 16-bit MFMA) or 16 (four fp32 MFMAs)
  constexpr int BNC = 16 * CF;             // columns per block
  static_assert(BT || CF == 2 || CF == 4, "[K, N] B is read two or four columns per lane");
  constexpr int kFrag = NB * MF * CF;
  constexpr int kParts = F32 ? 2 : 1;  // fp32: totals and compensations
  constexpr int kTile = MF * 16 * (BNC + 4);
  constexpr int kTree = WV / 2 * kFrag * kParts * 256;
  __shared__ __attribute__((aligned(16))) float lds[kTree > NB * kTile ? kTree : NB * kTile];
  if (skip_item(ep)) return;
  batch_bases(A, B0, C, ep);
  const int n0 = blockIdx.x * BNC, m0 = blockIdx.y * (MF * 16);
  const int lane = lane_id(), w = wave_id();
  const int i16 = lane & 15, g = lane >> 4;
  const S* Bm[2] = {B0, B1};

  // Rows past M (columns past N of [N, K] B) re-read the last one; their results are not stored.
  const S* pa[MF];
#pragma unroll
  for (int i = 0; i < MF; ++i) pa[i] = A + (int64_t)min(m0 + i * 16 + i16, M - 1) * lda + g * KV;
  int64_t ob[BT ? CF : 1];
  const int ncol = n0 + VN * i16;  // [K, N] B: this lane's first column
  if constexpr (BT) {
#pragma unroll
    for (int c = 0; c < CF; ++c) ob[c] = (int64_t)min(n0 + c * 16 + i16, N - 1) * ldb + g * KV;
  } else {
    ob[0] = (int64_t)(g * KV) * ldb + min(ncol, N - 1);
  }
  const bool nfull = BT || ncol + VN <= N;

  struct Group {
    u32x4 a[U][MF];
    u32x4 b[BT ? U : 1][NB][BT ? CF : 1];
    typename SV::R n[BT ? 1 : U][NB][BT ? 1 : KV];
  };
  auto load = [&](int k0, Group& x) {
    if (K - k0 >= U * KS) {  // uniform (k0 + U * KS may pass an int)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * KS;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if constexpr (BT) {
#pragma unroll
            for (int c = 0; c < CF; ++c) x.b[u][b][c] = *reinterpret_cast<const typename SV::V16*>(Bm[b] + ob[c] + k);
          } else {
#pragma unroll
            for (int r = 0; r < KV; ++r) {
              const S* p = Bm[b] + ob[0] + (int64_t)(k + r) * ldb;
              if (nfull) x.n[u][b][r] = reinterpret_cast<const typename SV::VR*>(p)->v;
              else x.n[u][b][r] = small_load_n<S, VN>(p, N - ncol);
            }
          }
        }
#pragma unroll
        for (int i = 0; i < MF; ++i) x.a[u][i] = *reinterpret_cast<const typename SV::V16*>(pa[i] + k);
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * KS, left = K - (k + g * KV);  // of this lane's KV
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if constexpr (BT) {
#pragma unroll
            for (int c = 0; c < CF; ++c) x.b[u][b][c] = small_load_k(Bm[b] + ob[c] + k, left);
          } else {
#pragma unroll
            for (int r = 0; r < KV; ++r)
              x.n[u][b][r] = small_load_n<S, VN>(Bm[b] + ob[0] + (int64_t)(k + r) * ldb, r < left ? N - ncol : 0);
          }
        }
#pragma unroll
        for (int i = 0; i < MF; ++i) x.a[u][i] = small_load_k(pa[i] + k, left);
      }
    }
  };

  f32x4 acc[NB][MF][CF], comp[F32 ? NB : 1][F32 ? MF : 1][F32 ? CF : 1];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
      for (int c = 0; c < CF; ++c) {
        acc[b][i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (F32) comp[b][i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  auto compute = [&](const Group& x) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int c = 0; c < CF; ++c) {
          u32x4 fb;
          if constexpr (BT) {
            fb = x.b[u][b][c];
          } else if constexpr (F32) {
#pragma unroll
            for (int r = 0; r < 4; ++r) fb[r] = x.n[u][b][r][c];
          } else {
            const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
            for (int p = 0; p < 4; ++p)
              fb[p] = __builtin_amdgcn_perm(x.n[u][b][2 * p + 1][c >> 1], x.n[u][b][2 * p][c >> 1], sel);
          }
#pragma unroll
          for (int i = 0; i < MF; ++i) {
            if constexpr (F32) {
              // 16 products from the negated compensation of the total, then Kahan's step
              f32x4 y = comp[b][i][c];
#pragma unroll
              for (int j = 0; j < 4; ++j)
                y = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(fb[j]), __uint_as_float(x.a[u][i][j]), y, 0, 0, 0);
              const f32x4 t = acc[b][i][c] + y;
#pragma unroll
              for (int e = 0; e < 4; ++e) comp[b][i][c][e] = kahan_bound(y[e] - (t[e] - acc[b][i][c][e]));
              acc[b][i][c] = t;
            } else {
              acc[b][i][c] = mfma16x16x32<T>(fb, x.a[u][i], acc[b][i][c]);
            }
          }
        }
  };
  // s + o; fp32: with what the total lost (two-sum) added to both compensations
  auto add = [&](f32x4& s, f32x4& sc, const f32x4& o, const f32x4& oc) {
    if constexpr (F32) {
      const f32x4 t = s + o, z = t - s;
      sc += oc + ((s - (t - z)) + (o - z));
      s = t;
    } else {
      s += o;
    }
  };
  constexpr int kGroup = U * KS, kStride = WV * LV * kGroup;
  int64_t k0 = (int64_t)w * kGroup;
  if constexpr (LV > 1) {
    // Slices in bit-reversed order, so that each pair the tree adds is complete before the next begins: level
    // d of part holds a finished left half of 2^d slices. Empty slices are added as the zeros they are.
    constexpr int LOG = LV == 4 ? 2 : 4;
    static_assert(LV == 1 << LOG && NB == 1, "four or sixteen slices of one product");
    f32x4 part[LOG][MF][CF], pcomp[LOG][F32 ? MF : 1][F32 ? CF : 1];
    auto slice_k = [&](int i) { return (int64_t)(w + WV * (int)(__builtin_bitreverse32((unsigned)i) >> (32 - LOG))) * kGroup; };
    auto finish = [&](int i) {
      bool held = false;
#pragma unroll
      for (int d = 0; d < LOG; ++d) {
        if (held) continue;
        held = ((i >> d) & 1) == 0;  // uniform
#pragma unroll
        for (int x = 0; x < MF; ++x)
#pragma unroll
          for (int c = 0; c < CF; ++c) {
            f32x4& s = part[d][x][c];
            f32x4& sc = pcomp[d][F32 ? x : 0][F32 ? c : 0];
            f32x4& ac = comp[0][F32 ? x : 0][F32 ? c : 0];
            if (held) {
              s = acc[0][x][c];
              acc[0][x][c] = f32x4{0.f, 0.f, 0.f, 0.f};
              if constexpr (F32) {
                sc = ac;
                ac = f32x4{0.f, 0.f, 0.f, 0.f};
              }
            } else {
              add(s, sc, acc[0][x][c], ac);
              acc[0][x][c] = s;
              if constexpr (F32) ac = sc;
            }
          }
      }
    };
    struct At {
      int i;
      int64_t k;
    };
    auto settle = [&](At a) {  // the first group at or after a
      while (a.k >= K) {
        if (++a.i == LV) break;
        a.k = slice_k(a.i);
      }
      return a;
    };
    int done = 0;
    At at = settle(At{0, slice_k(0)});
    if (at.i < LV) {
      Group x0, x1;
      load((int)at.k, x0);
      while (true) {
        At nx = settle(At{at.i, at.k + kStride});
        if (nx.i < LV) load((int)nx.k, x1);
        for (; done < at.i; ++done) finish(done);
        compute(x0);
        at = nx;
        if (at.i == LV) break;
        nx = settle(At{at.i, at.k + kStride});
        if (nx.i < LV) load((int)nx.k, x0);
        for (; done < at.i; ++done) finish(done);
        compute(x1);
        at = nx;
        if (at.i == LV) break;
      }
    }
    if (K > WV * kGroup)  // else each wave has one slice, and the others' zeros change nothing
      for (; done < LV; ++done) finish(done);
  } else if (k0 < K) {
    Group x0, x1;
    load((int)k0, x0);
    while (true) {
      const bool m1 = k0 + kStride < K;
      if (m1) load((int)k0 + kStride, x1);
      compute(x0);
      if (!m1) break;
      k0 += kStride;
      const bool m0 = k0 + kStride < K;
      if (m0) load((int)k0 + kStride, x0);
      compute(x1);
      if (!m0) break;
      k0 += kStride;
    }
  }

  // Tree over the waves: the upper half hands its sums to the lower half.
#pragma unroll
  for (int h = WV / 2; h > 0; h >>= 1) {
    f32x4* slot = reinterpret_cast<f32x4*>(lds) + (w & (h - 1)) * (kFrag * kParts * 64) + lane;
    if (w >= h && w < 2 * h) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int c = 0; c < CF; ++c) {
            const int f = (b * MF + i) * CF + c;
            slot[f * kParts * 64] = acc[b][i][c];
            if constexpr (F32) slot[(f * kParts + 1) * 64] = comp[b][i][c];
          }
    }
    __syncthreads();
    if (w < h) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int c = 0; c < CF; ++c) {
            const int f = (b * MF + i) * CF + c;
            if constexpr (F32) add(acc[b][i][c], comp[b][i][c], slot[f * kParts * 64], slot[(f * kParts + 1) * 64]);
            else add(acc[b][i][c], comp[0][0][0], slot[f * kParts * 64], comp[0][0][0]);
          }
    }
    __syncthreads();
  }

  // The block's tile, [m][n]: fragment c of a lane holds columns 16 c + 4 g + v ([N, K] B) or
  // CF (4 g + v) + c ([K, N] B) of row 16 i + i16.
  constexpr int P = BNC + 4;
  if (w == 0) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        float* t = lds + b * kTile + (i * 16 + i16) * P;
        if constexpr (F32) {  // the total plus what it lost (an overflowed total stays as it is)
#pragma unroll
          for (int c = 0; c < CF; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (fabsf(acc[b][i][c][v]) < INFINITY) acc[b][i][c][v] += comp[b][i][c][v];
        }
        if constexpr (BT) {
#pragma unroll
          for (int c = 0; c < CF; ++c) *reinterpret_cast<f32x4*>(t + 16 * c + 4 * g) = acc[b][i][c];
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int c = 0; c < CF; ++c) t[CF * (4 * g + v) + c] = acc[b][i][c][v];
        }
      }
  }
  __syncthreads();
  if (w >= MF) return;
  f32x4 out[NB][1][CF];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int c = 0; c < CF; ++c)
      out[b][0][c] = *reinterpret_cast<const f32x4*>(lds + b * kTile + (w * 16 + i16) * P + 16 * c + 4 * g);
  const int m = m0 + w * 16 + i16;
  if constexpr (F32) {
    if (m >= M) return;
    typedef f32x4 f32x4_u __attribute__((aligned(4)));
#pragma unroll
    for (int c = 0; c < CF; ++c) {
      f32x4 o = out[0][0][c];
      if constexpr (NB == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = gate_up<T, EPI>(o[e], out[1][0][c][e]);
      }
      const int n = n0 + 16 * c + 4 * g;
      float* q = C + (int64_t)m * ldc + n;
      if (n + 3 < N) {
        *reinterpret_cast<f32x4_u*>(q) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) q[e] = o[e];
      }
    }
  } else {
    tile_epilogue<T, NB, EPI, true, 1, CF>(C, B1, ldc, M, N, m, n0 + 4 * g, out, ep);
  }
}

template <typename T, bool BT, int NB, int EPI, int MF, int CF, int WV, int U, int LV = 1>
static void launch_small_cfg(const void* A, const void* B0, const void* B1, void* C, int M, int N, int K, int64_t lda,
                             int64_t ldb, int64_t ldc, hipStream_t s, const EpiArgs& ep) {
  using S = typename T::S;
  gemm_small<T, BT, NB, EPI, MF, CF, WV, LV, U><<<dim3((unsigned)cdiv(N, 16 * CF), (unsigned)cdiv(M, 16 * MF), ep.batch), WV * kWave, 0, s>>>(
      (const S*)A, (const S*)B0, (const S*)B1, (S*)C, M, N, K, lda, ldb, ldc, ep);
}

template <typename T, int NB, int EPI>
int launch_gemm_small(const void* A, const void* B0, const void* B1, void* C, int64_t M, int64_t N, int64_t K,
                      int64_t lda, int64_t ldb, int64_t ldc, bool bt, hipStream_t s, const EpiArgs& ep) {
#define AK_SM(BT, MF, CF, WV, U) \
  launch_small_cfg<T, BT, NB, EPI, MF, CF, WV, U>(A, B0, B1, C, (int)M, (int)N, (int)K, lda, ldb, ldc, s, ep)
  constexpr bool F32 = sizeof(typename T::S) == 4;
  if constexpr (NB == 1 && EPI == kEpiStore) {
    // A batch whose blocks pass the chip: four slices a wave on wider tiles, with the same sums (us, as one
    // product / so: f16 nt 16 x 128 x 512, 64 items 8.1 / 6.9, 512 items 40 / 19; nn 1 x 4096 x 4096, 8 items 92 / 52;
    // f32 nt 32 x 512 x 64, 64 items 20 / 16, 512 items 132 / 91). Not where that was no faster: f32 nt of few
    // rows and much k (8 x 768 x 768, 32 items 20 / 24), nn in groups of one k-step (32 x 3000 x 1000, 8 items 33 / 38).
    const int64_t blocks = N <= 4096 ? small_blocks(M, N, bt) * ep.batch : 0;
    const bool k64 = small_k64(M, N, bt);
    if (ep.batch > 1 && (F32 ? blocks > (bt ? 768 : 512) && !(bt && M <= 16 && K > 256) : blocks > 256 && (bt || k64))) {
#define AK_SMB(MF, CF, U)                                                                                             \
  if (bt) launch_small_cfg<T, true, 1, EPI, MF, CF, 4, U, 4>(A, B0, B1, C, (int)M, (int)N, (int)K, lda, ldb, ldc, s, ep); \
  else launch_small_cfg<T, false, 1, EPI, MF, CF, 4, U, 4>(A, B0, B1, C, (int)M, (int)N, (int)K, lda, ldb, ldc, s, ep)
      if (M <= 16) {
        AK_SMB(1, 4, 2);
      } else if (k64) {
        AK_SMB(2, 2, 2);
      } else {
        AK_SMB(2, 2, 1);
      }
#undef AK_SMB
      return record_launch();
    }
  }
  // Columns per block: few while N gives the chip few blocks (each block then walks K on 16 waves),
  // more for wide N, where the rows of A, re-read by every block, would cost as much as B.
  if (bt) {
    constexpr bool G = NB == 2;  // two B matrices: half the columns of each
    if (N <= 4096) {
      if (M <= 16 || N <= 1024) AK_SM(true, 1, 1, 16, 2);
      else if (M <= 32) AK_SM(true, 2, 1, 16, (G ? 1 : 2));
      else AK_SM(true, 2, (G ? 1 : 2), 16, 1);
    } else {
      if (M <= 16) AK_SM(true, 1, (G ? 2 : 4), 16, 1);
      else if (M <= 32) AK_SM(true, 2, (G ? 2 : 4), 8, 1);
      else AK_SM(true, 4, (G ? 1 : 2), 8, 1);
    }
    return record_launch();
  }
  if constexpr (NB == 1) {
    if (N <= 4096) {
      if (M <= 16 || N <= 1024) AK_SM(false, 1, 2, 16, 2);
      else AK_SM(false, 2, 2, 16, 1);
    } else {
      if (M <= 16) AK_SM(false, 1, 4, 8, 1);
      else if (M <= 32 || F32) AK_SM(false, 2, 4, 8, 1);
      else AK_SM(false, (F32 ? 2 : 4), 4, 8, 1);
    }
    return record_launch();
  }
#undef AK_SM
  return AK_EINVAL;
}

#define AK_SMALL_INST(T, NB, EPI)                                                                                  \
  template int launch_gemm_small<T, NB, EPI>(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, \
                                             int64_t, int64_t, int64_t, bool, hipStream_t, const EpiArgs&);
#define AK_SMALL_16(T)                \
  AK_SMALL_INST(T, 1, kEpiStore)      \
  AK_SMALL_INST(T, 1, kEpiResidual)   \
  AK_SMALL_INST(T, 1, kEpiRope)       \
  AK_SMALL_INST(T, 1, kEpiBias)       \
  AK_SMALL_INST(T, 1, kEpiBiasGelu)   \
  AK_SMALL_INST(T, 1, kEpiBiasResidual)
#define AK_SMALL_GU(T)            \
  AK_SMALL_INST(T, 2, kEpiSilu)   \
  AK_SMALL_INST(T, 2, kEpiGelu)   \
  AK_SMALL_INST(T, 2, kEpiRelu2)  \
  AK_SMALL_INST(T, 2, kEpiNone)
AK_SMALL_16(TF16)
AK_SMALL_16(TBF16)
AK_SMALL_INST(TF32, 1, kEpiStore)
AK_SMALL_GU(TF16)
AK_SMALL_GU(TBF16)
AK_SMALL_GU(TF32)

}  // namespace ak

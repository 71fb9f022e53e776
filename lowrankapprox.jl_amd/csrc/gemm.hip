// gemm.hip -- MFMA GEMM for the sketches and the factor products (gfx950).
//
// C (M x N) = alpha * op(A) (M x K) * op(B) (K x N) + beta * C, FP64 in and out.  Replaces the
// dgemm behind mul!(C, S, A) in the Gaussian sketch (src/sketch.jl:91-110) and the products of
// the factorizations.  Arithmetic (prec):
//   F64    v_mfma_f64_16x16x4f64, FP64 accumulate (the drop-in);
//   F32    operands rounded to FP32, v_mfma_f32_16x16x4f32, FP32 accumulate;
//   BF16   operands rounded to BF16, v_mfma_f32_16x16x32_bf16, FP32 accumulate;
//   BF16X3 each operand split into three BF16 terms (hi + mid + lo ~ 24 bits), the six
//          products of order <= 2 accumulated in FP32 (~FP32 accuracy at BF16 MFMA rate).
// Tiles are staged through LDS with k contiguous ([m][k] and [n][k]), so the sketch case
// (op(A) = Omega stored K x ell, op(B) = A stored K x N) is a straight copy; the next k-tile
// is prefetched into registers while the current one is multiplied.  Blocks that share a
// B tile (the M tiles of one N tile) are mapped to the same XCD so A is fetched once into
// that XCD's L2.  Split-K writes FP64 partials that a second kernel sums in fixed order.
#include "lra_internal.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <type_traits>
#include <condition_variable>
#include <mutex>
#include <set>
#include <tuple>
#include <vector>

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

template <int PREC> struct PT;
template <> struct PT<LRA_PREC_F64> { typedef double E; static const int P = 1; static const int BK = 16; static const int PAD = 1; };
template <> struct PT<LRA_PREC_F32> { typedef float E; static const int P = 1; static const int BK = 32; static const int PAD = 1; };
template <> struct PT<LRA_PREC_BF16> { typedef __bf16 E; static const int P = 1; static const int BK = 32; static const int PAD = 8; };
template <> struct PT<LRA_PREC_BF16X3> { typedef __bf16 E; static const int P = 3; static const int BK = 32; static const int PAD = 8; };

struct GemmDev {
  int M, N, K;
  double alpha, beta;
  const double* A; i64 lda; int transA;
  const double* B; i64 ldb; int transB;
  double* C; i64 ldc;
  const i64* bgather;
  double* partial;  // split-K partial sums [split][N][M]... laid out as split*(M*N) col-major M x N
  int splits, kchunk;
  int MT, NT, NG;  // M tiles, N tiles, groups (= NT * splits)
  int ct;          // store D(row, col) to C(col, row) (the transposed product, splits == 1)
};

__device__ __forceinline__ void split3(double x, __bf16* h, __bf16* m, __bf16* l) {
  const __bf16 hi = (__bf16)(float)x;
  const double r1 = x - (double)(float)hi;
  const __bf16 mi = (__bf16)(float)r1;
  const double r2 = r1 - (double)(float)mi;
  *h = hi; *m = mi; *l = (__bf16)(float)r2;
}

template <int PREC, int BM, int BN, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(256) void gemm_kernel(GemmDev p) {
  typedef typename PT<PREC>::E E;
  constexpr int P = PT<PREC>::P;
  constexpr int BK = PT<PREC>::BK;
  constexpr int LDK = BK + PT<PREC>::PAD;  // leading dimension (elements) of an LDS row
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int LA = BM * BK / 256;  // elements of A tile per thread
  constexpr int LB = BN * BK / 256;
  static_assert(WAVES_M * WAVES_N == 4, "4 waves");
  static_assert(LA * 256 == BM * BK && LB * 256 == BN * BK, "tile/threads");

  __shared__ E sA[P][BM * LDK];
  __shared__ E sB[P][BN * LDK];

  // ---- XCD-aware block -> (group, mt) mapping
  const int b = blockIdx.x;
  const int xcd = b & 7, idx = b >> 3;
  const int grp = (idx / p.MT) * 8 + xcd;
  const int mt = idx % p.MT;
  if (grp >= p.NG) return;
  const int nt = grp % p.NT, split = grp / p.NT;
  const int m0 = mt * BM, n0 = nt * BN;
  const int kbeg = split * p.kchunk;
  const int kend = min(p.K, kbeg + p.kchunk);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  // ---- staging map: thread loads LA elements of the A tile and LB of the B tile.
  // k-contiguous source (trans = 1 for A, 0 for B): element e -> (row r, k c) with k fastest.
  // m/n-contiguous source: element e -> row fastest.
  double ra[LA], rb[LB];
  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int t = 0; t < LA; ++t) {
      const int e = tid + 256 * t;
      int r, c;
      if (p.transA) { r = e / BK; c = e % BK; } else { r = e % BM; c = e / BM; }
      const int gm = m0 + r, gk = k0 + c;
      double v = 0.0;
      if (gm < p.M && gk < kend)
        v = p.transA ? p.A[gk + (i64)gm * p.lda] : p.A[gm + (i64)gk * p.lda];
      ra[t] = v;
    }
#pragma unroll
    for (int t = 0; t < LB; ++t) {
      const int e = tid + 256 * t;
      int r, c;
      if (!p.transB) { r = e / BK; c = e % BK; } else { r = e % BN; c = e / BN; }
      const int gn = n0 + r, gk = k0 + c;
      double v = 0.0;
      if (gn < p.N && gk < kend) {
        const i64 kk = p.bgather ? (p.bgather[gk] - 1) : gk;
        v = p.transB ? p.B[gn + kk * p.ldb] : p.B[kk + (i64)gn * p.ldb];
      }
      rb[t] = v;
    }
  };
  auto store_tiles = [&]() {
#pragma unroll
    for (int t = 0; t < LA; ++t) {
      const int e = tid + 256 * t;
      int r, c;
      if (p.transA) { r = e / BK; c = e % BK; } else { r = e % BM; c = e / BM; }
      const int o = r * LDK + c;
      if constexpr (PREC == LRA_PREC_BF16X3) {
        __bf16 h, mi, l;
        split3(ra[t], &h, &mi, &l);
        sA[0][o] = h; sA[1][o] = mi; sA[2][o] = l;
      } else if constexpr (PREC == LRA_PREC_BF16) {
        sA[0][o] = (__bf16)(float)ra[t];
      } else {
        sA[0][o] = (E)ra[t];
      }
    }
#pragma unroll
    for (int t = 0; t < LB; ++t) {
      const int e = tid + 256 * t;
      int r, c;
      if (!p.transB) { r = e / BK; c = e % BK; } else { r = e % BN; c = e / BN; }
      const int o = r * LDK + c;
      if constexpr (PREC == LRA_PREC_BF16X3) {
        __bf16 h, mi, l;
        split3(rb[t], &h, &mi, &l);
        sB[0][o] = h; sB[1][o] = mi; sB[2][o] = l;
      } else if constexpr (PREC == LRA_PREC_BF16) {
        sB[0][o] = (__bf16)(float)rb[t];
      } else {
        sB[0][o] = (E)rb[t];
      }
    }
  };

  typedef typename std::conditional<PREC == LRA_PREC_F64, d4, f4>::type AccT;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = AccT{0, 0, 0, 0};

  const int l16 = lane & 15, lq = lane >> 4;
  const int am0 = wm * WTM, bn0 = wn * WTN;

  auto compute = [&]() {
    if constexpr (PREC == LRA_PREC_F64 || PREC == LRA_PREC_F32) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        E af[TM], bfv[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[i] = sA[0][(am0 + i * 16 + l16) * LDK + kk + lq];
#pragma unroll
        for (int j = 0; j < TN; ++j) bfv[j] = sB[0][(bn0 + j * 16 + l16) * LDK + kk + lq];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (PREC == LRA_PREC_F64)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bfv[j], acc[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bfv[j], acc[i][j], 0, 0, 0);
          }
      }
    } else {
      // one 16x16x32 step per BK = 32
      bf8 af[P][TM], bfv[P][TN];
#pragma unroll
      for (int q = 0; q < P; ++q) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          af[q][i] = *reinterpret_cast<const bf8*>(&sA[q][(am0 + i * 16 + l16) * LDK + lq * 8]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          bfv[q][j] = *reinterpret_cast<const bf8*>(&sB[q][(bn0 + j * 16 + l16) * LDK + lq * 8]);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (PREC == LRA_PREC_BF16) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfv[0][j], acc[i][j], 0, 0, 0);
          } else {
            // smallest terms first: lo*hi, hi*lo, mid*mid, mid*hi, hi*mid, hi*hi
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[2][i], bfv[0][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfv[2][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bfv[1][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bfv[0][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfv[1][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfv[0][j], acc[i][j], 0, 0, 0);
          }
        }
    }
  };

  if (kbeg < kend) {
    load_tiles(kbeg);
    store_tiles();
    __syncthreads();
    for (int k0 = kbeg; k0 < kend; k0 += BK) {
      const bool more = k0 + BK < kend;
      if (more) load_tiles(k0 + BK);
      compute();
      __syncthreads();
      if (more) {
        store_tiles();
        __syncthreads();
      }
    }
  }

  // ---- epilogue.  Output lane layout of a 16x16 tile (column l16 in every case):
  //   f32/bf16 MFMA: register r holds row 4*lq + r;  f64 MFMA: register r holds row lq + 4*r.
  // With beta != 0 the C values of one row of tiles are loaded together (unconditional loads
  // from clamped addresses), so the epilogue waits for memory once per tile row.
  const bool rd = p.splits == 1 && p.beta != 0.0;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    double cv[TN][4];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + bn0 + j * 16 + l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + am0 + i * 16 + (PREC == LRA_PREC_F64 ? lq + 4 * r : lq * 4 + r);
        const bool ok = rd && row < p.M && col < p.N;
        const i64 ci = p.ct ? col + (i64)row * p.ldc : row + (i64)col * p.ldc;
        const double x = p.C[ok ? ci : 0];
        cv[j][r] = ok ? x : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + bn0 + j * 16 + l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + am0 + i * 16 + (PREC == LRA_PREC_F64 ? lq + 4 * r : lq * 4 + r);
        if (row < p.M && col < p.N) {
          const double v = (double)acc[i][j][r];
          if (p.splits > 1) {
            p.partial[(i64)split * p.M * p.N + row + (i64)col * p.M] = v;
          } else {
            const i64 ci = p.ct ? col + (i64)row * p.ldc : row + (i64)col * p.ldc;
            p.C[ci] = rd ? p.alpha * v + p.beta * cv[j][r] : p.alpha * v;
          }
        }
      }
    }
  }
}

// FP64 GEMM for the case where both operands are k-contiguous in memory (op(A) = A' with A
// stored K x M, op(B) = B stored K x N, no gather): the sketch B = Omega * A.  Every thread
// moves 16-byte pairs (two consecutive k) from HBM into registers two k-tiles ahead of the
// MFMAs, which consume the current one from one of two LDS buffers, so each k-tile costs one
// (LDS-only) barrier.  LDS rows hold BK = 16 doubles padded to 17, which keeps the 16 lanes of an MFMA
// operand read on distinct banks.
template <int BM, int BN, int WAVES_M, int WAVES_N, int BK = 16, bool F32 = false>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_kc_f64_kernel(GemmDev p) {
  // F32: the same FP64 loads, rounded to FP32 on the way into LDS, v_mfma_f32_16x16x4f32
  // with FP32 accumulation (the F32 sketch precision)
  using E = typename std::conditional<F32, float, double>::type;
  typedef float f4v __attribute__((ext_vector_type(4)));
  using ACC = typename std::conditional<F32, f4v, d4>::type;
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  constexpr int LDK = BK + 1, KP = BK / 2;  // KP: 16-byte k-pairs per tile row
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int CA = BM * KP, CB = BN * KP;  // 16-byte chunks per tile
  constexpr int LA = (CA + NT - 1) / NT, LB = (CB + NT - 1) / NT;
  __shared__ E sA[2][BM * LDK];
  __shared__ E sB[2][BN * LDK];

  const int b = blockIdx.x;
  const int xcd = b & 7, idx = b >> 3;
  const int grp = (idx / p.MT) * 8 + xcd;
  const int mt = idx % p.MT;
  if (grp >= p.NG) return;
  const int nt = grp % p.NT, split = grp / p.NT;
  const int m0 = mt * BM, n0 = nt * BN;
  const int kbeg = split * p.kchunk;
  const int kend = min(p.K, kbeg + p.kchunk);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  typedef double d2 __attribute__((ext_vector_type(2)));
  // (8-byte aligned: an odd leading dimension; still one 16-byte load)
  typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
  // chunk e of a tile -> (row e / KP, k pair e % KP).  Rows past M (columns past N) are read from
  // the last one, and chunks past the tile from its last: unconditional loads, so the wait for
  // one tile's registers leaves the loads of the next in flight.  What they put in the tile
  // reaches only outputs that are not stored.
  const double *pa[LA], *pb[LB];
  int oa[LA], ob[LB];
#pragma unroll
  for (int t = 0; t < LA; ++t) {
    const int e = min(tid + NT * t, CA - 1), r = e / KP, c = (e % KP) * 2;
    pa[t] = p.A + kbeg + c + (i64)min(m0 + r, p.M - 1) * p.lda;
    oa[t] = r * LDK + c;
  }
#pragma unroll
  for (int t = 0; t < LB; ++t) {
    const int e = min(tid + NT * t, CB - 1), r = e / KP, c = (e % KP) * 2;
    pb[t] = p.B + kbeg + c + (i64)min(n0 + r, p.N - 1) * p.ldb;
    ob[t] = r * LDK + c;
  }
  auto load_tiles = [&](d2 (&ra)[LA], d2 (&rb)[LB], int tile) {
    const i64 o = (i64)tile * BK;
#pragma unroll
    for (int t = 0; t < LA; ++t) ra[t] = *reinterpret_cast<const d2u*>(pa[t] + o);
#pragma unroll
    for (int t = 0; t < LB; ++t) rb[t] = *reinterpret_cast<const d2u*>(pb[t] + o);
  };
  // the last tile when the range does not end on one: k beyond the range is zero
  auto load_tail = [&](d2 (&ra)[LA], d2 (&rb)[LB], int tile) {
    const int left = kend - kbeg - tile * BK;
    const i64 o = (i64)tile * BK;
    auto get = [&](const double* src, int c) {
      d2 v = {0.0, 0.0};
      if (c + 1 < left) v = *reinterpret_cast<const d2u*>(src);
      else if (c < left) v.x = src[0];
      return v;
    };
#pragma unroll
    for (int t = 0; t < LA; ++t) ra[t] = get(pa[t] + o, oa[t] % LDK);
#pragma unroll
    for (int t = 0; t < LB; ++t) rb[t] = get(pb[t] + o, ob[t] % LDK);
  };
  auto store_tiles = [&](const d2 (&ra)[LA], const d2 (&rb)[LB], int buf) {
#pragma unroll
    for (int t = 0; t < LA; ++t) {
      if (CA % NT == 0 || tid + NT * t < CA) {
        sA[buf][oa[t]] = (E)ra[t].x;
        sA[buf][oa[t] + 1] = (E)ra[t].y;
      }
    }
#pragma unroll
    for (int t = 0; t < LB; ++t) {
      if (CB % NT == 0 || tid + NT * t < CB) {
        sB[buf][ob[t]] = (E)rb[t].x;
        sB[buf][ob[t] + 1] = (E)rb[t].y;
      }
    }
  };

  ACC acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = ACC{0, 0, 0, 0};
  const int l16 = lane & 15, lq = lane >> 4;
  const int am0 = wm * WTM, bn0 = wn * WTN;
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      E af[TM], bfv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = sA[buf][(am0 + i * 16 + l16) * LDK + kk + lq];
#pragma unroll
      for (int j = 0; j < TN; ++j) bfv[j] = sB[buf][(bn0 + j * 16 + l16) * LDK + kk + lq];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (F32)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bfv[j], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bfv[j], acc[i][j], 0, 0, 0);
        }
    }
  };
  // F32: the running sums are folded into a second set every 512 k, so that a long K range rounds
  // no more than a short one (relative error of a 136-row sketch of 8192 x 8192 in four ranges of
  // 2048: 8.1e-7 unfolded, 4.1e-7 folded; eight ranges of 1024 unfolded: 5.7e-7)
  constexpr int FOLD = 512 / (2 * BK);  // loop passes (of two tiles) between folds
  constexpr int FM = F32 ? TM : 1, FN = F32 ? TN : 1;
  ACC sum[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) sum[i][j] = ACC{0, 0, 0, 0};
  auto fold = [&] {
    if constexpr (F32) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = ACC{0, 0, 0, 0};
        }
    }
  };
  // waits for this wave's LDS operations, not for its global loads
  auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // (kbeg and c are even: a pair is on 16 bytes where its column is, else on 8)
  const int full = kbeg < kend ? (kend - kbeg) / BK : 0;
  int cur = 0;
  if (full > 0) {
    d2 ra0[LA], rb0[LB], ra1[LA], rb1[LB];  // tiles in flight, in turn
    load_tiles(ra0, rb0, 0);
    load_tiles(ra1, rb1, min(1, full - 1));
    store_tiles(ra0, rb0, 0);
    lds_barrier();
    // a tile's loads are issued two tiles before its MFMAs
    for (int t = 0; t < full; t += 2) {
      load_tiles(ra0, rb0, min(t + 2, full - 1));
      compute(0);
      store_tiles(ra1, rb1, 1);
      lds_barrier();
      cur = 1;
      if (t + 1 >= full) break;
      if (F32 && (t / 2) % FOLD == FOLD - 1) fold();
      load_tiles(ra1, rb1, min(t + 3, full - 1));
      compute(1);
      store_tiles(ra0, rb0, 0);
      lds_barrier();
      cur = 0;
    }
  }
  if (kbeg + full * BK < kend) {
    // (buffer `cur` is free: every wave is past the barrier after its last reads)
    d2 ra[LA], rb[LB];
    load_tail(ra, rb, full);
    store_tiles(ra, rb, cur);
    lds_barrier();
    compute(cur);
  }
  if constexpr (F32) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += sum[i][j];
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + bn0 + j * 16 + l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // f64 MFMA: register r holds row lq + 4 r; f32 MFMA: row 4 lq + r
        const int row = m0 + am0 + i * 16 + (F32 ? 4 * lq + r : lq + 4 * r);
        if (row < p.M && col < p.N) {
          const double v = (double)acc[i][j][r];
          if (p.splits > 1) {
            p.partial[(i64)split * p.M * p.N + row + (i64)col * p.M] = v;
          } else {
            double* c = p.C + row + (i64)col * p.ldc;
            *c = (p.beta == 0.0) ? p.alpha * v : p.alpha * v + p.beta * *c;
          }
        }
      }
    }
}

// C (M x N) = alpha op(A) op(B) + beta C, FP64, any storage order, for products whose 128 x 128
// tiles would be few (the blocked QR's X -= V W, a factor's Q times its small core): 16 rows by 64
// columns a wave, operands straight into the MFMA registers 16 k ahead, no LDS.  The product is
// formed transposed, D = op(B)' op(A)', so that 16 lanes hold 16 consecutive rows of a column of
// C.  Bound by reading and writing C for a short K (5689 x 199 at K = 32: 10 us, tiled 58: 90
// workgroups), by L1 reads of op(B) for a long one (5689 x 300 at K = 231: 50 us, tiled 132).  The
// k of an MFMA are 4 j + 0..3 in turn, the tiled kernel's order, so both give the same bits.
__global__ __launch_bounds__(256) void gemm_direct_kernel(int M, int N, int K,
                                                           const double* __restrict__ A, i64 am,
                                                           i64 ak, const double* __restrict__ B,
                                                           i64 bk, i64 bn, double alpha, double beta,
                                                           double* __restrict__ C, i64 ldc) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  const int m = (int)blockIdx.x * 64 + wave * 16 + l16, n0 = (int)blockIdx.y * 64;
  const double* pa = A + (i64)min(m, M - 1) * am;
  const double* pb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) pb[j] = B + (i64)min(n0 + 16 * j + l16, N - 1) * bn;
  // register r of tile j is column n0 + 16 j + q + 4 r
  double c[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + 16 * j + q + 4 * r;
      const bool ok = beta != 0.0 && m < M && n < N;
      const double x = C[ok ? m + (i64)n * ldc : 0];
      c[j][r] = ok ? x : 0.0;
    }
  d4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = d4{0, 0, 0, 0};
  double a[4], b[4][4];  // the next 16 k
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + 4 * u + q;
      const i64 kc = min(k, K - 1);  // (loaded in range, zero from K on)
      const double xa = pa[kc * ak];
      a[u] = k < K ? xa : 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double xb = pb[j][kc * bk];
        b[j][u] = k < K ? xb : 0.0;
      }
    }
  };
  load(0);
  for (int k0 = 0; k0 < K; k0 += 16) {
    double ca[4], cb[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ca[u] = a[u];
#pragma unroll
      for (int j = 0; j < 4; ++j) cb[j][u] = b[j][u];
    }
    if (k0 + 16 < K) load(k0 + 16);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(cb[j][u], ca[u], acc[j], 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + 16 * j + q + 4 * r;
      if (m < M && n < N)
        C[m + (i64)n * ldc] = beta != 0.0 ? alpha * acc[j][r] + beta * c[j][r] : alpha * acc[j][r];
    }
}

// C (M x N <= 16 NT) = alpha op(A) op(B) + beta C, FP64, one 32-row tile and one K range per
// workgroup; each wave takes every fourth 16-deep step of the range and the four partial tiles
// meet in LDS.  Operands go from memory to the MFMA registers: with k = 4 q + r for register r of
// lane quarter q, a lane reads four consecutive k of a k-contiguous operand (32 bytes), or one row
// of 16 lanes each of four k of an m-contiguous one (128 bytes).  A is read once; B (at most 64
// columns) comes from L1/L2.  The next step's operands load during the current step's MFMAs.
// Bound by the MFMAs and the reading of A in turn: 64 columns on 8192 x 436 (m-contiguous) take
// 24 us a call (213 by the tiled kernel), on 436 x 7756 with beta = 1 32 us (215), on their
// transposes 35 (43) and 30 us (132); 16 columns 17, 21, 20 and 16 us.
typedef double d2a8 __attribute__((ext_vector_type(2), aligned(8)));

template <int TA, int TB, int NT>
__global__ __launch_bounds__(256) void gemm_narrow_kernel(
    int M, int N, int K, int kchunk, const double* __restrict__ A, i64 lda,
    const double* __restrict__ B, i64 ldb, double* __restrict__ part, double alpha, double beta,
    double* __restrict__ C, i64 ldc) {
  __shared__ double red[4][32][16 * NT + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const int m0 = (int)blockIdx.x * 32, n0 = (int)blockIdx.z * 16 * NT;
  const int k0 = (int)blockIdx.y * kchunk, k1 = min(K, k0 + kchunk);
  const double* pa[2];
  const double* pb[NT];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const i64 m = min(m0 + 16 * i + l16, M - 1);
    pa[i] = TA ? A + m * lda : A + m;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const i64 n = min(n0 + 16 * j + l16, N - 1);
    pb[j] = TB ? B + n : B + n * ldb;
  }
  auto load4 = [&](const double* p, int contiguous, i64 ld, int k, double* v) {
    if (k + 16 - 4 * q <= k1) {  // the whole step is in range (the same for every lane)
      if (contiguous) {
        const d2a8 a = *reinterpret_cast<const d2a8*>(p + k);
        const d2a8 b = *reinterpret_cast<const d2a8*>(p + k + 2);
        v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = p[(i64)(k + r) * ld];
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const i64 kk = min(k + r, k1 - 1);
        const double x = p[contiguous ? kk : kk * ld];
        v[r] = k + r < k1 ? x : 0.0;
      }
    }
  };
  double a[2][4], b[NT][4];
  auto load = [&](int k) {
#pragma unroll
    for (int i = 0; i < 2; ++i) load4(pa[i], TA, lda, k + 4 * q, a[i]);
#pragma unroll
    for (int j = 0; j < NT; ++j) load4(pb[j], !TB, ldb, k + 4 * q, b[j]);
  };
  d4 acc[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = d4{0, 0, 0, 0};
  int k = k0 + 16 * wave;
  if (k < k1) load(k);
  for (; k < k1; k += 64) {
    double ca[2][4], cb[NT][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int i = 0; i < 2; ++i) ca[i][r] = a[i][r];
#pragma unroll
      for (int j = 0; j < NT; ++j) cb[j][r] = b[j][r];
    }
    if (k + 64 < k1) load(k + 64);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[i][r], cb[j][r], acc[i][j], 0, 0, 0);
  }
  // register r holds row q + 4 r of its tile
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][16 * i + q + 4 * r][16 * j + l16] = acc[i][j][r];
  __syncthreads();
  for (int e = tid; e < 32 * 16 * NT; e += 256) {
    const int row = e & 31, cl = e >> 5, col = n0 + cl;
    const i64 m = m0 + row;
    if (m >= M || col >= N) continue;
    const double v = (red[0][row][cl] + red[1][row][cl]) + (red[2][row][cl] + red[3][row][cl]);
    if (part) {
      part[(i64)blockIdx.y * M * N + m + (i64)col * M] = v;
    } else {
      double* c = C + m + (i64)col * ldc;
      *c = beta == 0.0 ? alpha * v : alpha * v + beta * *c;
    }
  }
}

__global__ void splitk_reduce_kernel(int M, int N, int splits, const double* part, double alpha,
                                     double beta, double* C, i64 ldc) {
  const i64 total = (i64)M * N;
  for (i64 e = blockIdx.x * (i64)blockDim.x + threadIdx.x; e < total;
       e += (i64)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int q = 0; q < splits; ++q) s += part[(i64)q * total + e];
    const i64 row = e % M, col = e / M;
    double* c = C + row + col * ldc;
    *c = (beta == 0.0) ? alpha * s : alpha * s + beta * *c;
  }
}

// C (M x N) = alpha A' B + beta C for a short product over a long K (M <= 32): the Gram-type
// products of the blocked QR (V'V and V'X, K = the panel's rows).  A workgroup owns a 32 x 32
// output tile and one K-range; 32-deep k-tiles of both operands are loaded coalesced (32
// consecutive k of one column per 32 lanes) into double-buffered LDS and consumed by
// v_mfma_f64_16x16x4f64, a 16 x 16 quarter per wave.  With several K-ranges the partials go
// to `part` ([split][M x N]) and splitk_reduce_kernel adds them in a fixed order.

__global__ __launch_bounds__(256) void gemm_tn_skinny_kernel(int M, int N, int K, int kchunk,
                                                             int ntiles, const double* __restrict__ A,
                                                             i64 lda, const double* __restrict__ B,
                                                             i64 ldb, double* __restrict__ part,
                                                             double alpha, double beta,
                                                             double* __restrict__ C, i64 ldc) {
  __shared__ double sA[2][32][33];  // [i][k]
  __shared__ double sB[2][32][33];  // [j][k]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nt = blockIdx.x % ntiles, split = blockIdx.x / ntiles;
  const int n0 = nt * 32;
  const int kbeg = split * kchunk, kend = min(K, kbeg + kchunk);
  const int kk = tid & 31, c0 = tid >> 5;  // loader: k offset, first column (+8 u)
  double ra[4], rb[4];
  auto load = [&](int k0) {
    const int k = k0 + kk;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = c0 + 8 * u;
      // unconditional loads from clamped addresses, masked afterwards
      const bool oa = k < kend && c < M, ob = k < kend && n0 + c < N;
      const double xa = A[oa ? k + (i64)c * lda : 0];
      const double xb = B[ob ? k + (i64)(n0 + c) * ldb : 0];
      ra[u] = oa ? xa : 0.0;
      rb[u] = ob ? xb : 0.0;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sA[buf][c0 + 8 * u][kk] = ra[u];
      sB[buf][c0 + 8 * u][kk] = rb[u];
    }
  };
  const int wm = wave & 1, wn = wave >> 1;
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  int buf = 0;
  if (kbeg < kend) {
    load(kbeg);
    store(0);
  }
  __syncthreads();
  for (int k0 = kbeg; k0 < kend; k0 += 32) {
    const bool more = k0 + 32 < kend;
    if (more) load(k0 + 32);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const double a = sA[buf][wm * 16 + (lane & 15)][ks * 4 + (lane >> 4)];
      const double b = sB[buf][wn * 16 + (lane & 15)][ks * 4 + (lane >> 4)];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
    if (more) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  // lane holds D(row = (lane >> 4) + 4 r, col = lane & 15) of its quarter
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = wm * 16 + (lane >> 4) + 4 * r, col = n0 + wn * 16 + (lane & 15);
    if (row >= M || col >= N) continue;
    if (part) {
      part[(i64)split * M * N + row + (i64)col * M] = acc[r];
    } else {
      double* c = C + row + (i64)col * ldc;
      *c = (beta == 0.0) ? alpha * acc[r] : alpha * acc[r] + beta * *c;
    }
  }
}

// ---- configurations -------------------------------------------------------------------
struct Cfg { int id, BM, BN; };
// id -> (BM, BN, WAVES_M, WAVES_N)
static const Cfg kCfgs[] = {{0, 16, 256}, {1, 32, 256}, {2, 48, 256}, {3, 64, 256}, {4, 128, 128},
                            {5, 16, 256}, {6, 32, 256}, {7, 48, 256}, {8, 64, 256}, {9, 128, 128},
                            {10, 64, 128}, {11, 128, 256}, {12, 128, 128}, {13, 64, 256},
                            {14, 256, 128}, {15, 80, 256}, {16, 96, 256}, {17, 160, 256},
                            {18, 176, 128}, {19, 208, 128}, {20, 112, 128}, {21, 112, 256},
                            {22, 144, 128}, {23, 144, 128}, {24, 112, 128}, {25, 48, 128}};
constexpr int kNumCfg = 26;
// ids 5..21: the k-contiguous kernel (gemm_kc_f64_kernel, FP64 or F32 MFMA; 11, 13, 14, 16-21
// with 512 threads, 12 with 32-wide k-tiles).  15-17 hold a short sketch (ell = 72, 136) in one
// M-tile, so each k-tile of A is read from L2 once; 18 (11 MFMA rows per wave) covers
// ell = 520 in three M-tiles with 1.5% padding; 19 (13 MFMA rows per wave) covers two paired
// rounds' 400 rows (orders 136 + 264) in two M-tiles, 20 and 21 the 112 rows of orders 40 + 72
// in one.
bool kc_cfg(int id) { return id >= 5; }
bool kc_aligned(const GemmArgs& g) {  // k pairs of both operands on 16 bytes
  return (g.lda % 2) == 0 && (g.ldb % 2) == 0 && ((uintptr_t)g.A % 16) == 0 &&
         ((uintptr_t)g.B % 16) == 0;
}
// g.odd: the sketches take it with operands on 8 bytes too (order
// 400 of 5689 x 2048 671 us on the generic tiles, 371 here; order 112 187 and 107).  The products inside the
// factorizations, and pheig's sketches, keep the generic tiles and their rounding.
bool kc_ok(const GemmArgs& g) {
  return (g.prec == LRA_PREC_F64 || g.prec == LRA_PREC_F32) && g.transA == 1 && g.transB == 0 &&
         g.bgather == nullptr && (g.odd || kc_aligned(g));
}
// Which kernels a product may take: products of one shape but different classes are tuned apart,
// since a configuration found for one may not be another's.  0: the generic tiles only, 1: the
// k-contiguous kernel too, 2: the k-contiguous kernel with operands on 8 bytes.
int kc_class(const GemmArgs& g) { return !kc_ok(g) ? 0 : kc_aligned(g) ? 1 : 2; }

template <int PREC>
hipError_t launch_cfg(int id, const GemmDev& d, int blocks, hipStream_t st) {
  switch (id) {
    case 0: hipLaunchKernelGGL((gemm_kernel<PREC, 16, 256, 1, 4>), dim3(blocks), dim3(256), 0, st, d); break;
    case 1: hipLaunchKernelGGL((gemm_kernel<PREC, 32, 256, 1, 4>), dim3(blocks), dim3(256), 0, st, d); break;
    case 2: hipLaunchKernelGGL((gemm_kernel<PREC, 48, 256, 1, 4>), dim3(blocks), dim3(256), 0, st, d); break;
    case 3: hipLaunchKernelGGL((gemm_kernel<PREC, 64, 256, 1, 4>), dim3(blocks), dim3(256), 0, st, d); break;
    case 4: hipLaunchKernelGGL((gemm_kernel<PREC, 128, 128, 2, 2>), dim3(blocks), dim3(256), 0, st, d); break;
    case 5:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<16, 256, 1, 4, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<16, 256, 1, 4, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 6:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<32, 256, 1, 4, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<32, 256, 1, 4, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 7:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<48, 256, 1, 4, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<48, 256, 1, 4, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 8:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 256, 1, 4, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 256, 1, 4, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 9:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 128, 2, 2, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 128, 2, 2, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 10:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 128, 2, 2, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 128, 2, 2, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 11:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 256, 2, 4, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 256, 2, 4, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 12:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 128, 2, 2, 32, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<128, 128, 2, 2, 32, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 13:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 256, 2, 4, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<64, 256, 2, 4, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 14:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<256, 128, 4, 2, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<256, 128, 4, 2, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 15:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<80, 256, 1, 4, 16, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<80, 256, 1, 4, 16, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 16:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<96, 256, 2, 4, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<96, 256, 2, 4, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 17:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<160, 256, 2, 4, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<160, 256, 2, 4, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 18:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<176, 128, 1, 8, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<176, 128, 1, 8, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 19:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<208, 128, 1, 8, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<208, 128, 1, 8, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 20:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 128, 1, 8, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 128, 1, 8, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 21:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 256, 1, 8, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 256, 1, 8, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 22:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<144, 128, 1, 8, 16, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<144, 128, 1, 8, 16, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 23:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<144, 128, 1, 8, 32, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<144, 128, 1, 8, 32, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 24:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 128, 1, 8, 32, false>), dim3(blocks), dim3(512), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<112, 128, 1, 8, 32, true>), dim3(blocks), dim3(512), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    case 25:
      if constexpr (PREC == LRA_PREC_F64) hipLaunchKernelGGL((gemm_kc_f64_kernel<48, 128, 1, 4, 32, false>), dim3(blocks), dim3(256), 0, st, d);
      else if constexpr (PREC == LRA_PREC_F32) hipLaunchKernelGGL((gemm_kc_f64_kernel<48, 128, 1, 4, 32, true>), dim3(blocks), dim3(256), 0, st, d);
      else return hipErrorInvalidValue;
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_prec(int prec, int id, const GemmDev& d, int blocks, hipStream_t st) {
  if (kc_cfg(id) && prec != LRA_PREC_F64 && prec != LRA_PREC_F32) return hipErrorInvalidValue;
  switch (prec) {
    case LRA_PREC_F64: return launch_cfg<LRA_PREC_F64>(id, d, blocks, st);
    case LRA_PREC_F32: return launch_cfg<LRA_PREC_F32>(id, d, blocks, st);
    case LRA_PREC_BF16: return launch_cfg<LRA_PREC_BF16>(id, d, blocks, st);
    case LRA_PREC_BF16X3: return launch_cfg<LRA_PREC_BF16X3>(id, d, blocks, st);
  }
  return hipErrorInvalidValue;
}

int bk_of(int prec) { return prec == LRA_PREC_F64 ? 16 : 32; }

// Autotuner: the first call for a shape class times every candidate (config, splits) on the
// live operands and caches the fastest; later calls reuse the choice.  The cache is
// process-wide and filled once per class: a call that finds the class being tuned by another
// thread (another context, e.g. a serving worker) waits for that choice instead of timing on
// its own, so every product of a class in the process uses one configuration and gives the
// same bits in any order and under any overlap.
struct TuneKey {
  int prec, transA, transB, mb, nb, kb, kc;
  bool operator<(const TuneKey& o) const {
    return std::tie(prec, transA, transB, mb, nb, kb, kc) <
           std::tie(o.prec, o.transA, o.transB, o.mb, o.nb, o.kb, o.kc);
  }
};
struct TuneVal { int cfg, splits; };
std::mutex g_tune_mu;
std::condition_variable g_tune_cv;
std::map<TuneKey, TuneVal> g_tune;
std::set<TuneKey> g_tuning;  // classes being tuned right now
int g_autotune = -1;

int bucket(i64 x) {  // power-of-two bucket
  int b = 0;
  while ((1ll << b) < x) ++b;
  return b;
}
// M's class: its 16-row MFMA tile count up to 1024 rows (a sketch order; the best M tile
// depends on how the order divides into tiles, e.g. 400 rows fill two 208-row tiles but
// 264 rows fit a 160 x 256 tile better), the power-of-two bucket beyond
int bucket_m(i64 m) { return m <= 1024 ? (int)((m + 15) / 16) : 64 + bucket(m); }

TuneKey key_of(const GemmArgs& g) {
  return {g.prec, g.transA, g.transB, bucket_m(g.M), bucket(g.N), bucket(g.K), kc_class(g)};
}

int prepare(lra_ctx* ctx, const GemmArgs& g, int cfg, int splits, GemmDev* d, int* blocks) {
  const Cfg& c = kCfgs[cfg];
  d->M = (int)g.M; d->N = (int)g.N; d->K = (int)g.K;
  d->alpha = g.alpha; d->beta = g.beta;
  d->A = g.A; d->lda = g.lda; d->transA = g.transA;
  d->B = g.B; d->ldb = g.ldb; d->transB = g.transB;
  d->C = g.C; d->ldc = g.ldc; d->bgather = g.bgather;
  const int bk = (cfg == 12 || (cfg >= 23 && cfg <= 25)) ? 32 : bk_of(g.prec);
  i64 kchunk = 0;
  if (g.K <= 0) {
    splits = 1;
  } else {
    kchunk = (g.K + splits - 1) / splits;
    kchunk = (kchunk + bk - 1) / bk * bk;
    splits = (int)((g.K + kchunk - 1) / kchunk);
  }
  d->splits = splits; d->kchunk = (int)kchunk;
  d->MT = (int)((g.M + c.BM - 1) / c.BM);
  d->NT = (int)((g.N + c.BN - 1) / c.BN);
  d->NG = d->NT * splits;
  d->partial = nullptr;
  d->ct = 0;
  if (splits > 1) {
    double* part = nullptr;
    LRA_CHECK(lra_wsT(ctx, WS_SPLITK, (size_t)splits * g.M * g.N, &part));
    d->partial = part;
  }
  const i64 groups8 = ((i64)d->NG + 7) / 8;
  const i64 nblk = groups8 * 8 * d->MT;
  if (nblk > 2147483647ll) { lra_set_error("gemm: grid too large"); return LRA_E_UNSUPPORTED; }
  *blocks = (int)nblk;
  return LRA_OK;
}

int run(lra_ctx* ctx, const GemmArgs& g, int cfg, int splits) {
  GemmDev d;
  int blocks = 0;
  LRA_CHECK(prepare(ctx, g, cfg, splits, &d, &blocks));
  hipError_t e = launch_prec(g.prec, cfg, d, blocks, ctx->stream);
  if (e != hipSuccess) {
    lra_set_error("gemm launch: %s", hipGetErrorString(e));
    return LRA_E_HIP;
  }
  if (d.splits > 1) {
    const i64 total = g.M * g.N;
    int rb = (int)std::min<i64>((total + 255) / 256, 16384);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(rb), dim3(256), 0, ctx->stream, (int)g.M,
                       (int)g.N, d.splits, d.partial, g.alpha, g.beta, g.C, g.ldc);
    e = hipGetLastError();
    if (e != hipSuccess) {
      lra_set_error("splitk reduce launch: %s", hipGetErrorString(e));
      return LRA_E_HIP;
    }
  }
  return LRA_OK;
}

// A' B with M <= 32 and a long K on gemm_tn_skinny_kernel: 32 x 32 tiles, K split so that
// about one workgroup per CU runs (ranges of at least 256, multiples of 32).
bool tn_skinny_ok(const GemmArgs& g) {
  return g.prec == LRA_PREC_F64 && g.transA == 1 && g.transB == 0 && g.bgather == nullptr &&
         g.M <= 32 && g.K >= 256;
}

int run_tn_skinny(lra_ctx* ctx, const GemmArgs& g) {
  const i64 ntiles = (g.N + 31) / 32;
  i64 splits = std::max<i64>(1, (ctx->num_cu + ntiles - 1) / ntiles);
  splits = std::min<i64>(splits, std::max<i64>(1, g.K / 256));
  i64 kchunk = (g.K + splits - 1) / splits;
  kchunk = (kchunk + 31) / 32 * 32;
  splits = (g.K + kchunk - 1) / kchunk;
  double* part = nullptr;
  if (splits > 1) LRA_CHECK(lra_wsT(ctx, WS_SPLITK, (size_t)(splits * g.M * g.N), &part));
  hipLaunchKernelGGL(gemm_tn_skinny_kernel, dim3((unsigned)(ntiles * splits)), dim3(256), 0,
                     ctx->stream, (int)g.M, (int)g.N, (int)g.K, (int)kchunk, (int)ntiles, g.A,
                     g.lda, g.B, g.ldb, part, g.alpha, g.beta, g.C, g.ldc);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && splits > 1) {
    const i64 total = g.M * g.N;
    const int rb = (int)std::min<i64>((total + 255) / 256, 16384);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(rb), dim3(256), 0, ctx->stream, (int)g.M,
                       (int)g.N, (int)splits, part, g.alpha, g.beta, g.C, g.ldc);
    e = hipGetLastError();
  }
  if (e != hipSuccess) {
    lra_set_error("skinny gemm launch: %s", hipGetErrorString(e));
    return LRA_E_HIP;
  }
  return LRA_OK;
}

// op(A) op(B) with few columns (a factor applied to a block of vectors) on gemm_narrow_kernel:
// 32 x 64 tiles whose four waves share K, K split further over workgroups (chunks of at least
// 128) until about two workgroups per CU run.  One pass over op(A) for every 64 columns, no LDS
// staging: the tiled kernels' 128-column tiles spend half or more of their MFMAs on padding, run
// on a few CUs (8192 x 436 by 64 columns: 64 workgroups) and are not tuned with beta != 0.
// Where the line lies (times of a call, tiled -> narrow): an operand that is not k-contiguous is
// read by narrow in any case up to 256 columns (8192 x 436: 224 -> 56 us at 256 columns, 8192 x
// 2048: 263 -> 201); with both k-contiguous the tuned tiles read it from LDS as well, and beyond
// 64 columns narrow is ahead only for short K (7756 x 436 at 128 columns 143 -> 48 us, 200 x
// 2000 34 -> 16, but 4096 x 4096 105 -> 121).
// The products inside the factorizations stay on the tiled kernels: a Hermitian factorization's
// eigenvectors take their signs from the rounding of its core, and the gain there is small
// (psvdfact of 5689 x 2048 13.5 -> 13.1 ms).
bool narrow_ok(const GemmArgs& g) {
  if (!g.narrow) return false;
  if (g.prec != LRA_PREC_F64 || g.bgather != nullptr || g.K < 1 || g.N > 256) return false;
  return g.N <= 64 || g.K <= 2048 || !kc_ok(g);
}

TuneVal heuristic(const GemmArgs& g, int num_cu);

int run_narrow(lra_ctx* ctx, const GemmArgs& g) {
  const i64 mt = (g.M + 31) / 32, nt = (g.N + 63) / 64, tiles = mt * nt;
  i64 splits = std::max<i64>(1, std::min<i64>((2 * ctx->num_cu + tiles - 1) / tiles, g.K / 128));
  // a context with a scratch limit: no more partial sums than the tiled kernels would take, or
  // than the slot holds already, so that what follows finds the room it needs
  if (ctx->hbm_budget != 0)
    splits = std::min<i64>(splits, std::max<i64>(heuristic(g, ctx->num_cu).splits,
                                                 (i64)(ctx->ws_size[WS_SPLITK] / sizeof(double)) /
                                                     (g.M * g.N)));
  i64 kchunk = (g.K + splits - 1) / splits;
  kchunk = (kchunk + 63) / 64 * 64;
  splits = (g.K + kchunk - 1) / kchunk;
  double* part = nullptr;
  if (splits > 1) {
    const int rc = lra_wsT(ctx, WS_SPLITK, (size_t)(splits * g.M * g.N), &part);
    if (rc == LRA_E_ALLOC) {  // a budget without room for the partial sums: one range
      splits = 1;
      kchunk = (g.K + 63) / 64 * 64;
    } else if (rc != LRA_OK) {
      return rc;
    }
  }
  const dim3 grid((unsigned)mt, (unsigned)splits, (unsigned)nt);
#define NARROW(TA, TB, NT)                                                                     \
  hipLaunchKernelGGL((gemm_narrow_kernel<TA, TB, NT>), grid, dim3(256), 0, ctx->stream,        \
                     (int)g.M, (int)g.N, (int)g.K, (int)kchunk, g.A, g.lda, g.B, g.ldb, part,  \
                     g.alpha, g.beta, g.C, g.ldc)
#define NARROW_T(NT)                                                                           \
  if (g.transA) { if (g.transB) NARROW(1, 1, NT); else NARROW(1, 0, NT); }                     \
  else { if (g.transB) NARROW(0, 1, NT); else NARROW(0, 0, NT); }
  if (g.N <= 16) { NARROW_T(1) }
  else if (g.N <= 32) { NARROW_T(2) }
  else { NARROW_T(4) }
#undef NARROW_T
#undef NARROW
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && splits > 1) {
    const int rb = (int)std::min<i64>((g.M * g.N + 255) / 256, 16384);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(rb), dim3(256), 0, ctx->stream, (int)g.M,
                       (int)g.N, (int)splits, part, g.alpha, g.beta, g.C, g.ldc);
    e = hipGetLastError();
  }
  if (e != hipSuccess) {
    lra_set_error("narrow gemm launch: %s", hipGetErrorString(e));
    return LRA_E_HIP;
  }
  return LRA_OK;
}

// Operands on 8 bytes get no more K ranges on the k-contiguous kernel's wider tiles than on the
// generic ones: the partial sums are scratch that a context may limit.
void candidates(const GemmArgs& g, int num_cu, std::vector<TuneVal>* out) {
  const bool kc = kc_ok(g), odd = kc_class(g) == 2;
  int generic = 1;
  for (int cfg = 0; cfg < kNumCfg; ++cfg) {
    const Cfg& c = kCfgs[cfg];
    if (kc_cfg(cfg) && !kc) continue;
    // skip configs that waste most of the M tile
    if (c.BM > 16 && g.M <= c.BM / 2) continue;
    if ((cfg == 4 || cfg == 9 || cfg == 11 || cfg == 12) && g.M < 96) continue;
    if (cfg == 14 && g.M < 192) continue;
    const i64 tiles = ((g.M + c.BM - 1) / c.BM) * ((g.N + c.BN - 1) / c.BN);
    for (int s : {1, 2, 3, 4, 6, 8, 16, 32}) {
      if (s > 1 && tiles * s > 8ll * num_cu) break;
      if (s > 1 && g.K / s < 256) break;
      if (!kc_cfg(cfg)) generic = std::max(generic, s);
      else if (odd && s > generic) break;
      out->push_back({cfg, s});
    }
  }
  if (out->empty()) out->push_back({4, 1});
}

TuneVal heuristic(const GemmArgs& g, int num_cu) {
  int cfg = 4;
  if (g.M <= 16) cfg = 0;
  else if (g.M <= 32) cfg = 1;
  else if (g.M <= 48) cfg = 2;
  else if (g.M <= 64) cfg = 3;
  const Cfg& c = kCfgs[cfg];
  const i64 tiles = ((g.M + c.BM - 1) / c.BM) * ((g.N + c.BN - 1) / c.BN);
  int s = 1;
  while (tiles * s < 2ll * num_cu && g.K / (2 * s) >= 512 && s < 32) s *= 2;
  return {cfg, s};
}

// Where gemm_direct_kernel takes a product of operands that are not both k-contiguous: up to 512 k
// (one K range in either form) and 2 M elements of C.  Tiled -> direct: 1817 x 300 at K = 231 66
// -> 29 us, 1000 x 1000 at K = 500 89 -> 61, 5689 x 300 (1.7 M) at K = 500 250 -> 103; 4000 x
// 1000 (4 M) at K = 231 75 -> 91.
bool direct_ok(const GemmArgs& g) {
  return g.prec == LRA_PREC_F64 && g.bgather == nullptr && g.K >= 1 && g.K <= 512 &&
         g.M * g.N <= (1ll << 21) && !(kc_ok(g) && kc_aligned(g));
}

int run_direct(lra_ctx* ctx, const GemmArgs& g) {
  const dim3 grid((unsigned)((g.M + 63) / 64), (unsigned)((g.N + 63) / 64));
  hipLaunchKernelGGL(gemm_direct_kernel, grid, dim3(256), 0, ctx->stream, (int)g.M, (int)g.N,
                     (int)g.K, g.A, g.transA ? g.lda : 1, g.transA ? 1 : g.lda, g.B,
                     g.transB ? g.ldb : 1, g.transB ? 1 : g.ldb, g.alpha, g.beta, g.C, g.ldc);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    lra_set_error("direct gemm launch: %s", hipGetErrorString(e));
    return LRA_E_HIP;
  }
  return LRA_OK;
}

// A short-K product with a tall C (the blocked QR's X -= V W and its like): formed as the
// transposed product C' = op(B)' op(A)' stored transposed, so that the MFMA output tile puts 16
// consecutive rows of one column of C in 16 consecutive lanes and the read-modify-write of C is
// coalesced.  One K-range, the general kernel's configuration for the swapped shape.
bool ct_ok(const GemmArgs& g) {
  return g.bgather == nullptr && g.K <= 64 && g.M >= 256 && g.M >= 2 * g.N;
}
// In FP64 gemm_direct_kernel takes it (with the same bits) up to 2 M elements of C, where the tiles
// are few; beyond, only where op(B) is read along its columns or K is short; and with at most 32
// columns, half its tile or more idle, up to 32768 rows.  Tiled -> direct: 5689 x 16 at K = 32
// 9.2 -> 6.3 us, 4096 x 512 at K = 64 29 -> 18 to 26, 8192 x 2048 at K = 8 68 -> 50, with op(B) = B'
// at K = 64 108 -> 85, but with op(B) = B at K = 32 82 -> 94 and 16384 x 4096 306 -> 450; 30000 x 32
// at K = 32 13.5 -> 10.7, 60000 x 32 14.7 -> 18.8 and x 16 10.0 -> 15.3.
bool ct_direct(const GemmArgs& g) {
  if (g.prec != LRA_PREC_F64 || g.K < 1) return false;
  if (g.N <= 32) return g.M <= 32768;
  return g.M * g.N <= (1ll << 21) || g.transB || (g.K <= 16 && g.M * g.N <= (1ll << 25));
}

int run_ct(lra_ctx* ctx, const GemmArgs& g) {
  if (ct_direct(g)) return run_direct(ctx, g);
  GemmArgs s = g;
  s.M = g.N; s.N = g.M;
  s.A = g.B; s.lda = g.ldb; s.transA = !g.transB;
  s.B = g.A; s.ldb = g.lda; s.transB = !g.transA;
  const int cfg = heuristic(s, ctx->num_cu).cfg;
  GemmDev d;
  int blocks = 0;
  LRA_CHECK(prepare(ctx, s, cfg, 1, &d, &blocks));
  d.C = g.C; d.ldc = g.ldc;
  d.ct = 1;
  const hipError_t e = launch_prec(g.prec, cfg, d, blocks, ctx->stream);
  if (e != hipSuccess) {
    lra_set_error("gemm launch: %s", hipGetErrorString(e));
    return LRA_E_HIP;
  }
  return LRA_OK;
}

}  // namespace

int lra_gemm(lra_ctx* ctx, const GemmArgs& g) {
  if (g.M <= 0 || g.N <= 0) return LRA_OK;
  if (g.M > 2147483647ll || g.N > 2147483647ll || g.K > 2147483647ll) {
    lra_set_error("gemm: dimension exceeds int32");
    return LRA_E_UNSUPPORTED;
  }
  if (g_autotune < 0) {
    const char* env = getenv("LRA_AUTOTUNE");
    g_autotune = (env && env[0] == '0') ? 0 : 1;
  }
  // LRA_GEMM_CFG=id:splits forces a configuration (when it applies to the operands)
  if (const char* f = getenv("LRA_GEMM_CFG")) {
    int id = -1, sp = 1;
    if (sscanf(f, "%d:%d", &id, &sp) == 2 && id >= 0 && id < kNumCfg && sp >= 1 &&
        (!kc_cfg(id) || kc_ok(g)))
      return run(ctx, g, id, sp);
  }
  if (tn_skinny_ok(g)) return run_tn_skinny(ctx, g);
  if (ct_ok(g)) return run_ct(ctx, g);
  if (narrow_ok(g)) return run_narrow(ctx, g);
  if (direct_ok(g)) return run_direct(ctx, g);
  const TuneKey key = key_of(g);
  TuneVal choice;
  bool have = false;
  {
    std::unique_lock<std::mutex> lk(g_tune_mu);
    for (;;) {
      auto it = g_tune.find(key);
      if (it != g_tune.end()) { choice = it->second; have = true; break; }
      if (!g_tuning.count(key)) { g_tuning.insert(key); break; }  // this call tunes it
      g_tune_cv.wait(lk);
    }
  }
  if (!have) {
    // (on an error return the class is released so that a later call tunes it)
    struct Release {
      const TuneKey& k;
      bool armed = true;
      ~Release() {
        if (!armed) return;
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tuning.erase(k);
        g_tune_cv.notify_all();
      }
    } release{key};
    if (!g_autotune || g.beta != 0.0 || (g.M * g.N * (g.K > 0 ? g.K : 1)) < (1ll << 24)) {
      choice = heuristic(g, ctx->num_cu);
    } else {
      std::vector<TuneVal> cands;
      candidates(g, ctx->num_cu, &cands);
      hipEvent_t e0, e1;
      LRA_HIP(hipEventCreate(&e0));
      LRA_HIP(hipEventCreate(&e1));
      auto time_of = [&](const TuneVal& c, int reps, float* ms) -> int {
        LRA_HIP(hipEventRecord(e0, ctx->stream));
        for (int r = 0; r < reps; ++r) LRA_CHECK(run(ctx, g, c.cfg, c.splits));
        LRA_HIP(hipEventRecord(e1, ctx->stream));
        LRA_HIP(hipEventSynchronize(e1));
        LRA_HIP(hipEventElapsedTime(ms, e0, e1));
        *ms /= (float)reps;
        return LRA_OK;
      };
      // pass 1: every candidate once warm + 2 timed; pass 2: the four fastest re-timed twice
      // more, 3 launches each, interleaved, so a single noisy timing does not pick the tile
      std::vector<std::pair<float, int>> t1;
      for (size_t i = 0; i < cands.size(); ++i) {
        LRA_CHECK(run(ctx, g, cands[i].cfg, cands[i].splits));  // warm
        float ms = 0.f;
        LRA_CHECK(time_of(cands[i], 2, &ms));
        t1.push_back({ms, (int)i});
      }
      std::sort(t1.begin(), t1.end());
      const size_t top = std::min<size_t>(4, t1.size());
      std::vector<float> best_of(top);
      for (size_t i = 0; i < top; ++i) best_of[i] = t1[i].first;
      for (int pass = 0; pass < 2; ++pass)
        for (size_t i = 0; i < top; ++i) {
          float ms = 0.f;
          LRA_CHECK(time_of(cands[t1[i].second], 3, &ms));
          best_of[i] = std::min(best_of[i], ms);
        }
      size_t win = 0;
      for (size_t i = 1; i < top; ++i)
        if (best_of[i] < best_of[win]) win = i;
      choice = cands[t1[win].second];
      hipEventDestroy(e0);
      hipEventDestroy(e1);
    }
    {
      std::lock_guard<std::mutex> lk(g_tune_mu);
      g_tune[key] = choice;
      g_tuning.erase(key);
      release.armed = false;
    }
    g_tune_cv.notify_all();
  }
  return run(ctx, g, choice.cfg, choice.splits);
}

// Report the configuration chosen for a sketch's shape with operands on 16 bytes (for the bench's
// roofline bookkeeping).  LRA_E_STATE: not tuned yet, or a shape whose kernel is not tuned.
extern "C" int lra_gemm_choice(int prec, int transA, int transB, int64_t M, int64_t N,
                               int64_t K, int* cfg, int* splits, int* bm, int* bn) {
  GemmArgs g{};
  g.M = M; g.N = N; g.K = K;
  g.transA = transA; g.transB = transB; g.prec = prec;
  g.lda = g.ldb = 2;  // (even, as the null pointers: aligned)
  if (tn_skinny_ok(g) || ct_ok(g) || direct_ok(g)) return LRA_E_STATE;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tune.find(key_of(g));
  if (it == g_tune.end()) return LRA_E_STATE;
  *cfg = it->second.cfg;
  *splits = it->second.splits;
  *bm = kCfgs[it->second.cfg].BM;
  *bn = kCfgs[it->second.cfg].BN;
  return LRA_OK;
}

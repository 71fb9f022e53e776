// qrcp_block.hip -- blocks of pivoted-QR steps for sketches in HBM.
//
// A single step (qg_fused) reads and writes the whole trailing matrix for one reflector: at
// 2056 x 3758 that is 24 us a step.  Here a block of up to 16 pivots is found first, without
// touching the trailing matrix, and then applied to it in one pass:
//   qb_select  one workgroup: LAPACK's bookkeeping of the block just applied (dlaqps block ends,
//              stop rule, per step), then the (at most) 128 trailing columns of largest norm as
//              candidates and the largest norm outside them;
//   qb_gram    the candidates' Gram matrix on the rows not yet factored (MFMA);
//   qb_panel   one workgroup: pivoted Cholesky of that matrix picks the pivots in order, then the
//              Householder QR of the picked columns (rows in registers);
//   qb_apply   16 trailing columns per workgroup, held in registers in MFMA layout: W = V'A and
//              V'V, A -= V (T'W), then the block's norm downdates (LAWN 176), column by column.
// The pivots are those of the step-by-step factorization: column norms only fall, so a
// candidate whose residual norm (from the Cholesky) exceeds every norm outside the candidates
// is the largest of all.  A block ends where that no longer holds, and before the Gram matrix
// loses accuracy: residual squares below 1e-2 of the block's first.  The reflectors themselves
// come from the columns (dlarfg), never from the Gram matrix.  The downdates replay each step
// of the block from the rows of R with LAPACK's test (the block's own pivots included, up to
// their step); a recomputed norm at step t is the norm at the block's end plus the rows of R in
// between, so the dlaqps block ends fall on the same steps as step by step.
//
// Measured on a 2056 x 3758 sketch of sigma_i = exp(-0.01 (i-1)), 1152 steps in 128 blocks:
// 10.2 ms against 26.9 ms of single steps.  A block at s = 500 takes 80 us: select 6 and gram 11
// (latency: dependent loads of one workgroup, and 2300 rows over 16 waves), panel 32 (the chain
// of pivots, 0.7 us each, and of columns, 1.6 us each), apply 32 (reading and writing the
// trailing matrix at about 5 TB/s).  128 candidates because their Gram matrix fits LDS, where a
// pivot costs one row read; 16 columns because V and the tiles of the apply are then one MFMA
// tile wide and the panel's rows fit one workgroup's registers.
#include "lra_qg.h"
#include "lra_wave.h"

#include <algorithm>
#include <climits>

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
// two consecutive doubles of a column: 8-byte aligned (any step, any leading dimension)
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef double d2v __attribute__((ext_vector_type(2)));

constexpr int QT = 1024;  // threads of every kernel here

// ---- bookkeeping and candidates ---------------------------------------------------------

// VPT positions per thread in registers (n <= 1024 VPT), else read three times (VPT = 0).
// Bound by its chain of dependent loads and barriers: the norms load while thread 0 does the
// bookkeeping, each wave reduces the waves' maxima itself, and only norms of at least half the
// largest enter the histogram (256 bins, one wave's scan).  Every wave reads step, length and
// `done` from the state on entry, so thread 0 keeps their new values until the barrier after the
// bookkeeping: every wave's entry reads are behind it.
template <int VPT>
__global__ __launch_bounds__(QT) void qb_select(int n, int kmax, int nb, int stop_after,
                                                const double* __restrict__ vn1,
                                                const double* __restrict__ diag, int* at,
                                                int* cand, FState* st) {
  constexpr int NW = QT / 64, NBIN = 256;
  __shared__ int s_done, s_cnt, s_T;
  __shared__ double s_mx[NW], s_tau[NW];
  __shared__ int s_mp[NW];
  __shared__ int hist[NBIN];
  if (st->done) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int s0 = st->s, b = st->b, s = s0 + b;  // (unless the block holds the last step)
  auto norm_at = [&](int p) {
    const double x = vn1[at[p]];
    return x >= 0.0 ? x : -1.0;  // (a NaN norm takes no part)
  };
  double v[VPT ? VPT : 1];
  int c[VPT ? VPT : 1];
  if constexpr (VPT > 0) {
#pragma unroll
    for (int r = 0; r < VPT; ++r) {
      const int p = s + tid + r * QT;
      c[r] = p < n ? at[p] : -1;
    }
#pragma unroll
    for (int r = 0; r < VPT; ++r) {
      const double x = c[r] >= 0 ? vn1[c[r]] : -1.0;
      v[r] = x >= 0.0 ? x : -1.0;
    }
  }
  if (tid < NBIN) hist[tid] = 0;
  int done = 0, e = b;  // (thread 0's)
  if (tid == 0) {
    const unsigned mask = st->mask;
    if (b > 0) {
      int j0 = st->j0, jb = st->jb;
      for (int t = 0; t < b && !done; ++t) {
        const int step = s0 + t, s1 = step + 1;
        if (!((step - j0 + 1 == jb) || ((mask >> t) & 1) || s1 == kmax)) continue;
        const double ptol = st->ptol;
        bool stop = false;
        if (fabs(diag[step]) <= ptol) {
          int i = j0;
          for (; i < step; ++i)
            if (fabs(diag[i]) <= ptol) break;
          st->k = i;
          stop = true;
        }
        if (!stop && s1 == kmax) { st->k = kmax; stop = true; }
        if (!stop && stop_after > 0 && s1 >= stop_after) {
          st->k = s1;
          st->early = 1;
          stop = true;
        }
        if (stop) {
          done = 1;
          e = t + 1;
        } else {
          j0 = s1;
          jb = min(nb, kmax - s1);
        }
      }
      st->j0 = j0;
      st->jb = jb;
      // the swaps of steps after the one that stopped are taken back, last first
      const int* swp = cand + 2 * QB_C;
      for (int t = b - 1; t >= e; --t) {
        const int p = swp[t], cc = at[s0 + t];
        at[s0 + t] = at[p];
        at[p] = cc;
      }
    }
    s_done = done;
    s_cnt = 0;
    s_T = NBIN;
  }
  // the largest norm, lowest position first among equals
  double bv = -1.0;
  int bp = INT_MAX;
  if constexpr (VPT > 0) {
#pragma unroll
    for (int r = 0; r < VPT; ++r)
      if (v[r] > bv) { bv = v[r]; bp = s + tid + r * QT; }
  } else {
    for (int p = s + tid; p < n; p += QT) {
      const double x = norm_at(p);
      if (x > bv) { bv = x; bp = p; }
    }
  }
  double wv;
  const int wl = wave_argmax(bv, bp, 1, &wv);
  const int wp = __builtin_amdgcn_readlane(bp, wl < 0 ? 0 : wl);
  if (lane == 0) {
    s_mx[wave] = wv;
    s_mp[wave] = wl < 0 ? INT_MAX : wp;
  }
  __syncthreads();
  if (tid == 0) {
    st->s = s0 + e;
    st->b = 0;
    st->mask = 0;
    st->sprev = -1;
    st->done = done;
  }
  if (s_done) return;
  const double lv = lane < NW ? s_mx[lane] : -1.0;
  const int lp = lane < NW ? s_mp[lane] : INT_MAX;
  double vmax;
  const int ml = wave_argmax(lv, lp, 1, &vmax);
  if (ml < 0) {  // no candidate (NaN norms)
    if (tid == 0) {
      st->k = s;
      st->done = 1;
    }
    return;
  }
  const int ap = __builtin_amdgcn_readlane(lp, ml);
  if (tid == 0) {
    cand[0] = at[ap];
    cand[QB_C] = ap;
  }
  // squares of norms outside this range do not fit the Gram matrix: single steps
  if (!(vmax >= 1e-140 && vmax <= 1e140)) {
    if (tid == 0) st->ncand = 0;
    return;
  }
  // bin of a norm: 256 bins from half the largest to the largest, -1 below
  const double sc = 2.0 * NBIN / vmax;
  auto bin_of = [&](double x) { return x * 2.0 >= vmax ? min(NBIN - 1, (int)(x * sc) - NBIN) : -1; };
  auto count = [&](double x) {
    const int k = bin_of(x);
    if (k >= 0) atomicAdd(&hist[k], 1);
  };
  if constexpr (VPT > 0) {
#pragma unroll
    for (int r = 0; r < VPT; ++r) count(v[r]);
  } else {
    for (int p = s + tid; p < n; p += QT) count(norm_at(p));
  }
  __syncthreads();
  // the lowest bin T with at most QB_C - 1 columns in the bins from T up
  if (wave == 0) {
    int h[4], tot = 0;
#pragma unroll
    for (int k = 3; k >= 0; --k) {
      h[k] = hist[4 * lane + k];
      tot += h[k];
    }
    int up = tot;  // columns in this lane's bins and all above
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_down(up, d, 64);
      if (lane + d < 64) up += o;
    }
    up -= tot;
    if (up < QB_C) {
#pragma unroll
      for (int k = 3; k >= 0; --k) {
        if (up < QB_C && up + h[k] >= QB_C) s_T = 4 * lane + k + 1;  // (one lane at the most)
        up += h[k];
      }
      if (lane == 0 && up < QB_C) s_T = 0;
    }
  }
  __syncthreads();
  const int T = s_T;
  double tau = -1.0;
  auto place = [&](double x, int p, int col) {
    if (p == ap || x < 0.0) return;
    if (bin_of(x) >= T) {
      const int i = 1 + atomicAdd(&s_cnt, 1);
      cand[i] = col;
      cand[QB_C + i] = p;
    } else {
      tau = fmax(tau, x);
    }
  };
  if constexpr (VPT > 0) {
#pragma unroll
    for (int r = 0; r < VPT; ++r) place(v[r], s + tid + r * QT, c[r]);
  } else {
    for (int p = s + tid; p < n; p += QT) place(norm_at(p), p, at[p]);
  }
  tau = wave_max(tau);
  if (lane == 0) s_tau[wave] = tau;
  __syncthreads();
  if (wave == 0) {
    tau = wave_max(lane < NW ? s_tau[lane] : -1.0);
    if (lane == 0) {
      st->tau = tau;
      st->ncand = min(QB_C, 1 + s_cnt);
    }
  }
}

// the pivot of step s (candidate 0) moved to position s, for single steps that follow
__global__ void qb_pick_kernel(const int* cand, int* at, const FState* st) {
  if (st->done) return;
  const int s = st->s, p = cand[QB_C];
  if (p != s) {
    const int c = at[s];
    at[s] = cand[0];
    at[p] = c;
  }
}

// The block's downdates of one column's norm (a, a2: vn1, vn2), steps 0 .. steps - 1, row t of
// the column's R at R[t * ldr]; tail: the squares of its rows from `steps` on.  Returns the mask
// of the steps after which LAPACK recomputes the norm (and ends its block).
__device__ __forceinline__ unsigned downdate(double& a, double& a2, const double* R, int ldr,
                                             int steps, double tail, int s, int lastrk) {
  const double tol3z = 1.0536712127723509e-08;  // sqrt(dlamch('E'))
  unsigned mask = 0;
  for (int t = 0; t < steps; ++t) {
    if (s + t + 1 >= lastrk || a == 0.0) continue;
    double temp = fabs(R[t * ldr]) / a;
    temp = (1.0 + temp) * (1.0 - temp);
    temp = temp < 0.0 ? 0.0 : temp;
    const double r = a / a2;
    if (temp * r * r <= tol3z) {
      double sum = tail;
      for (int i = steps - 1; i > t; --i) sum += R[i * ldr] * R[i * ldr];
      a = a2 = sqrt(sum);
      mask |= 1u << t;
    } else {
      a *= sqrt(temp);
    }
  }
  return mask;
}

// ---- Gram matrix of the candidates -------------------------------------------------------

// four rows r0 .. r0 + 3 of a column (zero from `rows` on)
__device__ __forceinline__ d4 load4(const double* __restrict__ c, int r0, int rows, bool full) {
  d4 x;
  if (full) {
    const d2u a = *reinterpret_cast<const d2u*>(c + r0), b = *reinterpret_cast<const d2u*>(c + r0 + 2);
    x = d4{a.x, a.y, b.x, b.y};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = r0 + r < rows ? c[r0 + r] : 0.0;
  }
  return x;
}

// One workgroup per 16 x 16 tile (ti >= tj) of the 8 x 8 tiles; its waves share the rows.
__global__ __launch_bounds__(QT) void qb_gram(int m, const double* __restrict__ B, i64 ldb,
                                              const int* __restrict__ cand, double* __restrict__ G,
                                              const FState* st) {
  __shared__ double red[QT / 64][256];
  if (st->done) return;
  const int nc = st->ncand;
  int ti = 0, tj = blockIdx.x;
  while (tj > ti) { tj -= ti + 1; ++ti; }
  if (16 * ti >= nc || nc < 2) return;
  const int s = st->s, rows = m - s, ntile = (rows + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, l16 = lane & 15;
  const double* ca = B + (i64)cand[min(16 * ti + l16, nc - 1)] * ldb + s;
  const double* cb = B + (i64)cand[min(16 * tj + l16, nc - 1)] * ldb + s;
  d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 3
  for (int t = wave; t < ntile; t += QT / 64) {
    const bool full = 16 * t + 16 <= rows;
    const d4 a = load4(ca, 16 * t + 4 * q, rows, full), b = load4(cb, 16 * t + 4 * q, rows, full);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b[r], acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][(q + 4 * r) * 16 + l16] = acc[r];
  __syncthreads();
  if (tid >= 256) return;
  double v = 0.0;
#pragma unroll
  for (int w = 0; w < QT / 64; ++w) v += red[w][tid];
  const int i = 16 * ti + tid / 16, j = 16 * tj + tid % 16;
  G[i * QB_C + j] = v;
  if (ti != tj) G[j * QB_C + i] = v;
}

// ---- pivots and panel --------------------------------------------------------------------

constexpr int QB_RED = 2 * (QT / 64) * QB_B;  // doubles of the panel's reductions
constexpr size_t kPanelLds = (size_t)QB_C * QB_C * 8 + (size_t)QB_RED * 8 + 2 * QB_B * 8 + 512;

// v_permlane32_swap / v_permlane16_swap on doubles: the upper half (odd 16-lane rows) of a and
// the lower half (even rows) of b change places, so a + b afterwards is a's sum in the lower
// half (even rows) and b's in the other.
__device__ __forceinline__ double swap_add32(double a, double b) {
  const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}
__device__ __forceinline__ double swap_add16(double a, double b) {
  const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}

// Step t of the panel's Householder QR: x is row tid + QT q of every column.
template <int t, int RP, int NB>
__device__ __forceinline__ void panel_step(double (&x)[RP][NB], int b, double* red, double* prow,
                                           double* s_tau, double* tau, double* diag) {
  if (t >= b) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, qt = lane >> 4;
  constexpr int par = t & 1;
  double* rd = red + par * (QT / 64) * QB_B;
  // dots of column t below row t with the block's columns from t on, four at a time: two lane
  // swaps leave column j0 + {0, 2, 1, 3}[row of 16 lanes] to sum over its 16 lanes
#pragma unroll
  for (int j0 = t; j0 < NB; j0 += 4) {
    if (j0 < b) {
      double p[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        p[u] = 0.0;
        if (j0 + u < NB) {
#pragma unroll
          for (int q = 0; q < RP; ++q) {
            const double xt = (q > 0 || tid > t) ? x[q][t] : 0.0;
            p[u] += xt * x[q][j0 + u < NB ? j0 + u : t];
          }
        }
      }
      const double w = group_sum(swap_add16(swap_add32(p[0], p[1]), swap_add32(p[2], p[3])), 16);
      const int j = j0 + (qt == 1 ? 2 : (qt == 2 ? 1 : qt));
      if (l16 == 0 && j < NB) rd[wave * QB_B + j] = w;
    }
  }
  if (tid == t) {
#pragma unroll
    for (int j = t; j < NB; ++j) prow[par * QB_B + j] = x[0][j];
  }
  __syncthreads();
  double sj = 0.0;
  const bool mine = l16 >= t && l16 < b;
  if (mine) {
#pragma unroll
    for (int w = 0; w < 4; ++w) sj += rd[(4 * qt + w) * QB_B + l16];
  }
  sj = swap_add16(sj, sj);
  sj = swap_add32(sj, sj);
  const double pj = mine ? prow[par * QB_B + l16] : 0.0;
  const double alpha = readlane_f64(pj, t), xn2 = readlane_f64(sj, t);
  double beta = alpha, tu = 0.0, scal = 0.0;
  if (xn2 != 0.0) {
    // (no rescaling as in dlarfg: the block's norms are between 1e-141 and 1e140)
    beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
    tu = (beta - alpha) / beta;
    scal = 1.0 / (alpha - beta);
  }
  const double wj = tu * (pj + sj * scal);
  double v[RP];
#pragma unroll
  for (int q = 0; q < RP; ++q)
    v[q] = (q > 0 || tid > t) ? x[q][t] * scal : (tid == t ? 1.0 : 0.0);
#pragma unroll
  for (int j = t + 1; j < NB; ++j) {
    if (j < b) {
      const double w = readlane_f64(wj, j);
#pragma unroll
      for (int q = 0; q < RP; ++q) x[q][j] -= w * v[q];
    }
  }
#pragma unroll
  for (int q = 0; q < RP; ++q)
    if (q > 0 || tid > t) x[q][t] = v[q];
  if (tid == t) x[0][t] = beta;
  if (tid == 0) {
    tau[t] = tu;
    diag[t] = beta;
    s_tau[t] = tu;
  }
}

// RP rows per thread, at most NB columns.
template <int RP, int NB>
__global__ __launch_bounds__(QT) void qb_panel(int m, int n, int kmax, double* __restrict__ B,
                                               i64 ldb, int* at, double* tau, double* diag,
                                               int* cand, const double* __restrict__ G,
                                               const double* __restrict__ vn1,
                                               const double* __restrict__ vn2,
                                               double* __restrict__ V, double* __restrict__ tb,
                                               int exact_tail, FState* st) {
  if (st->done) return;
  const int nc = st->ncand;
  if (nc < 1) return;
  extern __shared__ double lds[];
  double* sG = lds;                     // QB_C x QB_C
  double* red = sG + QB_C * QB_C;       // [parity][wave][column]
  double* prow = red + QB_RED;          // [parity][column]
  int* s_piv = (int*)(prow + 2 * QB_B);  // storage columns of the block
  int* s_b = s_piv + QB_B;
  double* s_tau = (double*)(s_b + 2);   // tau of the block (QB_B)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = st->s, rows = m - s;
  if (nc > 1) {
    // (entries beyond the candidates' 16-column tiles are not formed, and not used)
    d2v g[QB_C * QB_C / (2 * QT)];
#pragma unroll
    for (int e = 0; e < QB_C * QB_C / (2 * QT); ++e)
      g[e] = reinterpret_cast<const d2v*>(G)[tid + QT * e];
#pragma unroll
    for (int e = 0; e < QB_C * QB_C / (2 * QT); ++e)
      reinterpret_cast<d2v*>(sG)[tid + QT * e] = g[e];
  }
  __syncthreads();
  if (wave == 0) {
    const int bmax = min(NB, kmax - s);
    const int j0 = lane, j1 = lane + 64;
    double d0 = j0 < nc ? (nc > 1 ? sG[j0 * QB_C + j0] : 1.0) : -1.0;
    double d1 = j1 < nc ? sG[j1 * QB_C + j1] : -1.0;
    int p0 = j0 < nc ? cand[QB_C + j0] : INT_MAX, p1 = j1 < nc ? cand[QB_C + j1] : INT_MAX;
    int win = s + lane < n && lane < QB_B ? at[s + lane] : 0;  // at[s .. s + 15]
    const int c0 = j0 < nc ? cand[j0] : 0, c1 = j1 < nc ? cand[j1] : 0;
    const double tq = st->tau > 0.0 ? st->tau * (1.0 + 1e-9) : 0.0;
    double lim = tq * tq;  // a later pivot's residual square must exceed this
    if (exact_tail) {      // no step past a diagonal that could end the factorization
      const double pt = st->ptol * 1.01;
      lim = fmax(lim, pt * pt);
    }
    double first = 0.0;
    double L0[NB], L1[NB];
    int b = 0;
    bool go = true;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      if (!go || t >= bmax) { go = false; continue; }
      int lsel = 0, which = 0;
      if (t > 0) {
        const bool hi = d1 > d0 || (d1 == d0 && p1 < p0);
        const double bv = hi ? d1 : d0;
        double mx;
        const int w = wave_argmax(bv, hi ? p1 : p0, 1, &mx);
        if (w < 0 || !(mx > lim) || !(mx >= 1e-2 * first)) { go = false; continue; }
        lsel = w;
        which = __builtin_amdgcn_readlane(hi ? 1 : 0, w);
      }
      const int p = lsel + 64 * which;
      const double dp = readlane_f64(which ? d1 : d0, lsel);
      if (t == 0) first = dp;
      const int P = __builtin_amdgcn_readlane(which ? p1 : p0, lsel);
      const int col = __builtin_amdgcn_readlane(which ? c1 : c0, lsel);
      // LAPACK's swap of positions s + t and P (the window at[s .. s + 15] is in the lanes)
      const int occ = __builtin_amdgcn_readlane(win, t);
      if (P < s + QB_B) win = lane == P - s ? occ : win;
      else if (lane == 0) at[P] = occ;
      win = lane == t ? col : win;
      if (p0 == s + t) p0 = P;
      if (p1 == s + t) p1 = P;
      if (lane == 0) {
        s_piv[t] = col;
        cand[2 * QB_C + t] = P;
      }
      b = t + 1;
      if (nc > 1) {
        // 1 / sqrt(dp): the hardware estimate and two Newton steps (the values pick pivots,
        // they enter no result)
        double rs = __builtin_amdgcn_rsq(dp);
        rs = rs * (1.5 - (0.5 * dp * rs) * rs);
        rs = rs * (1.5 - (0.5 * dp * rs) * rs);
        double g0 = sG[p * QB_C + j0], g1 = sG[p * QB_C + j1];
#pragma unroll
        for (int i = 0; i < t; ++i) {
          const double lp = readlane_f64(which ? L1[i] : L0[i], lsel);
          g0 -= lp * L0[i];
          g1 -= lp * L1[i];
        }
        g0 *= rs;
        g1 *= rs;
        L0[t] = g0;
        L1[t] = g1;
        if (d0 >= 0.0) d0 = fmax(d0 - g0 * g0, 0.0);
        if (d1 >= 0.0) d1 = fmax(d1 - g1 * g1, 0.0);
      } else {
        go = false;
      }
      if (lane == lsel) {
        if (which) d1 = -1.0;
        else d0 = -1.0;
      }
    }
    if (lane < QB_B && s + lane < n) at[s + lane] = win;
    if (lane == 0) *s_b = b;
  }
  __syncthreads();
  const int b = *s_b;
  // the block's columns in registers: row tid + QT q of every column
  double x[RP][NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const double* c = B + (i64)(j < b ? s_piv[j] : s_piv[0]) * ldb + s;
#pragma unroll
    for (int q = 0; q < RP; ++q) {
      const int r = tid + QT * q;
      x[q][j] = (j < b && r < rows) ? c[r] : 0.0;
    }
  }
#define QB_STEP(t) if constexpr (t < NB) panel_step<t, RP, NB>(x, b, red, prow, s_tau, tau + s, diag + s);
  QB_STEP(0) QB_STEP(1) QB_STEP(2) QB_STEP(3) QB_STEP(4) QB_STEP(5) QB_STEP(6) QB_STEP(7)
  QB_STEP(8) QB_STEP(9) QB_STEP(10) QB_STEP(11) QB_STEP(12) QB_STEP(13) QB_STEP(14) QB_STEP(15)
#undef QB_STEP
  // R and the reflectors to the columns; V with its unit diagonal, zero above and past the block
  const int rpad = (rows + 15) / 16 * 16;
#pragma unroll
  for (int q = 0; q < RP; ++q) {
    const int r = tid + QT * q;
    if (r >= rpad) continue;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j < b && r < rows) B[(i64)s_piv[j] * ldb + s + r] = x[q][j];
    }
    double* vt = V + (i64)(r >> 4) * 256 + (r & 15);
#pragma unroll
    for (int j = 0; j < QB_B; ++j)
      vt[16 * j] = j < NB && j < b ? (r > j ? x[q][j < NB ? j : 0] : (r == j ? 1.0 : 0.0)) : 0.0;
  }
  if (tid < QB_B) tb[tid] = tid < b ? s_tau[tid] : 0.0;
  // a pivot's norm is downdated by the steps before its own, too: R to LDS, a lane per pivot
  double* sR = sG;  // [row][17]
  if (tid < QB_B) {
#pragma unroll
    for (int j = 0; j < NB; ++j) sR[tid * 17 + j] = x[0][j];
  }
  __syncthreads();
  if (tid < 64) {
    unsigned mask = 0;
    if (tid > 0 && tid < b) {
      const int lastrk = min(m, n), col = s_piv[tid];
      const double d = sR[tid * 17 + tid];  // |R(s + tid, s + tid)|: the rest of the column
      double a = vn1[col], a2 = vn2[col];
      mask = downdate(a, a2, sR + tid, 17, tid, d * d, s, lastrk);
    }
    for (int k = 1; k < 16; k <<= 1) mask |= (unsigned)__shfl_xor((int)mask, k, 16);
    if (tid == 0) {
      if (mask) st->mask = mask;  // (cleared by qb_select; qb_apply adds to it)
      st->b = b;
    }
  }
}

// ---- the block applied to the trailing columns -------------------------------------------

// RT row tiles of 16 per wave.  KEEP: the columns stay in registers between the two products
// (rows up to 256 RT); otherwise they are read twice.
template <int RT, bool KEEP>
__global__ __launch_bounds__(QT) void qb_apply(int m, int n, int lastrk, double* __restrict__ B,
                                               i64 ldb, const int* __restrict__ at, double* vn1,
                                               double* vn2, const double* __restrict__ V,
                                               const double* __restrict__ tau, FState* st) {
  __shared__ double red[QT / 64][256], red2[QT / 64][256], sV[256], sW[256];
  __shared__ double snrm[QT / 64][16], sR[16][17], sT[16];
  if (st->done) return;
  const int b = st->b, s = st->s;
  if (b == 0) return;
  const int pb = s + b + 16 * (int)blockIdx.x;
  if (pb >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, l16 = lane & 15;
  const bool have = pb + l16 < n;
  const int col = at[have ? pb + l16 : pb];
  double* c = B + (i64)col * ldb + s;
  const int rows = m - s, ntile = (rows + 15) / 16;
  if (tid < QB_B) sT[tid] = tau[tid];
  d4 x[KEEP ? RT : 1];
  // W = V'A and V'V in one pass over V (its second product hides behind the loads)
  d4 acc = {0.0, 0.0, 0.0, 0.0}, vv = {0.0, 0.0, 0.0, 0.0};
  auto dots = [&](int t, d4 y) {
    const double* vp = V + (i64)t * 256 + 16 * l16 + 4 * q;
    const d2v va = *reinterpret_cast<const d2v*>(vp), vb = *reinterpret_cast<const d2v*>(vp + 2);
    const double v[4] = {va.x, va.y, vb.x, vb.y};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[r], y[r], acc, 0, 0, 0);
      vv = __builtin_amdgcn_mfma_f64_16x16x4f64(v[r], v[r], vv, 0, 0, 0);
    }
  };
  if constexpr (KEEP) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int t = wave + (QT / 64) * i;
      if (t < ntile) x[i] = load4(c, 16 * t + 4 * q, rows, 16 * t + 16 <= rows);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int t = wave + (QT / 64) * i;
      if (t < ntile) dots(t, x[i]);
    }
  } else {
#pragma unroll 2
    for (int t = wave; t < ntile; t += QT / 64)
      dots(t, load4(c, 16 * t + 4 * q, rows, 16 * t + 16 <= rows));
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    red[wave][(q + 4 * r) * 16 + l16] = acc[r];
    red2[wave][(q + 4 * r) * 16 + l16] = vv[r];
  }
  __syncthreads();
  if (tid < 512) {
    const double(*rr)[256] = tid < 256 ? red : red2;
    double w = 0.0;
#pragma unroll
    for (int k = 0; k < QT / 64; ++k) w += rr[k][tid & 255];
    (tid < 256 ? sW : sV)[tid & 255] = w;
  }
  __syncthreads();
  // T'W without T: T^-1 = diag(1 / tau) + the strict upper triangle of V'V, so its transpose is
  // solved forward, w_i = tau_i (W_i - sum_{k < i} (V'V)_ki w_k), a lane per column
  if (tid < 16) {
    double w[QB_B];
#pragma unroll
    for (int i = 0; i < QB_B; ++i) {
      asm volatile("" ::: "memory");  // (one row's values at a time in registers)
      double a = sW[i * 16 + tid];
#pragma unroll
      for (int k = 0; k < i; ++k) a -= sV[k * 16 + i] * w[k];
      w[i] = sT[i] * a;
      red[0][i * 16 + tid] = -w[i];
    }
  }
  __syncthreads();
  double w2[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) w2[k] = red[0][(4 * k + q) * 16 + l16];
  // A - V (T'W): operand rows permuted so that the result's register r is row 4 q + r, as loaded
  const int vr = 4 * (l16 & 3) + (l16 >> 2);
  double ss = 0.0;
  auto update = [&](int t, d4 y) {
    const double* vp = V + (i64)t * 256 + vr;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      y = __builtin_amdgcn_mfma_f64_16x16x4f64(vp[16 * (4 * k + q)], w2[k], y, 0, 0, 0);
    const int r0 = 16 * t + 4 * q;
    if (have) {
      if (16 * t + 16 <= rows) {
        *reinterpret_cast<d2u*>(c + r0) = d2u{y[0], y[1]};
        *reinterpret_cast<d2u*>(c + r0 + 2) = d2u{y[2], y[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r0 + r < rows) c[r0 + r] = y[r];
      }
    }
    if (t == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sR[4 * q + r][l16] = y[r];
        ss += 4 * q + r >= b ? y[r] * y[r] : 0.0;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) ss += y[r] * y[r];
    }
  };
  if constexpr (KEEP) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int t = wave + (QT / 64) * i;
      if (t < ntile) update(t, x[i]);
    }
  } else {
#pragma unroll 2
    for (int t = wave; t < ntile; t += QT / 64)
      update(t, load4(c, 16 * t + 4 * q, rows, 16 * t + 16 <= rows));
  }
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (q == 0) snrm[wave][l16] = ss;
  __syncthreads();
  if (tid >= 16) return;
  unsigned mask = 0;
  if (have) {
    double tail = 0.0;
#pragma unroll
    for (int w = 0; w < QT / 64; ++w) tail += snrm[w][tid];
    double a = vn1[col], a2 = vn2[col];
    mask = downdate(a, a2, &sR[0][tid], 17, b, tail, s, lastrk);
    vn1[col] = a;
    vn2[col] = a2;
  }
  for (int d = 1; d < 16; d <<= 1) mask |= (unsigned)__shfl_xor((int)mask, d, 16);
  if (tid == 0 && mask) atomicOr(&st->mask, mask);
}

void launch_select(lra_ctx* c, const QrcpCall& q, const QbWork& w, const int* at, double* vn1,
                   const double* diag, FState* st) {
#define QS_ARGS dim3(1), dim3(QT), 0, c->stream, q.n, q.kmax, q.nb, q.stop_after, vn1, diag, \
                const_cast<int*>(at), w.cand, st
  if (q.n <= 4 * QT) hipLaunchKernelGGL(qb_select<4>, QS_ARGS);
  else if (q.n <= 8 * QT) hipLaunchKernelGGL(qb_select<8>, QS_ARGS);
  else if (q.n <= 16 * QT) hipLaunchKernelGGL(qb_select<16>, QS_ARGS);
  else hipLaunchKernelGGL(qb_select<0>, QS_ARGS);
#undef QS_ARGS
}

template <int RP, int NB>
void launch_panel(lra_ctx* c, const QrcpCall& q, const QbWork& w, int* at, const double* vn1,
                  const double* vn2, double* diag, FState* st) {
  static std::atomic<uint64_t> lds_set{0};
  lra_lds_limit_once(lds_set, (const void*)qb_panel<RP, NB>, (int)kPanelLds);
  hipLaunchKernelGGL((qb_panel<RP, NB>), dim3(1), dim3(QT), kPanelLds, c->stream, q.m, q.n, q.kmax,
                     q.A, q.lda, at, q.tau, diag, w.cand, w.G, vn1, vn2, w.V, w.T, q.exact_tail, st);
}

}  // namespace

QbWork lra_qb_work(double* w, int m) {
  QbWork o;
  o.cand = reinterpret_cast<int*>(w);  // 2 QB_C + 16 ints in QB_C + 16 doubles
  o.G = w + QB_C + 16;
  o.V = o.G + QB_C * QB_C;
  o.T = o.V + ((size_t)m + 31) / 16 * 256;
  return o;
}

int lra_qb_start(lra_ctx* c, const QrcpCall& q, const QbWork& w, const int* at, double* vn1,
                 const double* diag, FState* st) {
  launch_select(c, q, w, at, vn1, diag, st);
  LRA_HIP(hipGetLastError());
  return LRA_OK;
}

int lra_qb_pick(lra_ctx* c, const QbWork& w, int* at, FState* st) {
  hipLaunchKernelGGL(qb_pick_kernel, dim3(1), dim3(1), 0, c->stream, w.cand, at, st);
  LRA_HIP(hipGetLastError());
  return LRA_OK;
}

int lra_qb_blocks(lra_ctx* c, const QrcpCall& q, const QbWork& w, int* at, double* vn1,
                  double* vn2, double* diag, FState* st, int s, int count) {
  const int m = q.m, n = q.n, rows = m - s, lastrk = std::min(m, n);
  const unsigned ga = (unsigned)std::max(1, (n - s - 1 + 15) / 16);
  for (int k = 0; k < count; ++k) {
    hipLaunchKernelGGL(qb_gram, dim3(36), dim3(QT), 0, c->stream, m, q.A, q.lda, w.cand, w.G, st);
    // (the steps a panel holds: lra_qb_cap)
    if (rows <= QT) launch_panel<1, 16>(c, q, w, at, vn1, vn2, diag, st);
    else if (rows <= 2 * QT) launch_panel<2, 16>(c, q, w, at, vn1, vn2, diag, st);
    else if (rows <= 3 * QT) launch_panel<3, 12>(c, q, w, at, vn1, vn2, diag, st);
    else if (rows <= 4 * QT) launch_panel<4, 8>(c, q, w, at, vn1, vn2, diag, st);
    else launch_panel<8, 4>(c, q, w, at, vn1, vn2, diag, st);
#define QA_ARGS dim3(ga), dim3(QT), 0, c->stream, m, n, lastrk, q.A, q.lda, at, vn1, vn2, w.V, w.T, st
    if (rows <= 2 * 256) hipLaunchKernelGGL((qb_apply<2, true>), QA_ARGS);
    else if (rows <= 4 * 256) hipLaunchKernelGGL((qb_apply<4, true>), QA_ARGS);
    else if (rows <= 6 * 256) hipLaunchKernelGGL((qb_apply<6, true>), QA_ARGS);
    else if (rows <= 9 * 256) hipLaunchKernelGGL((qb_apply<9, true>), QA_ARGS);
    else hipLaunchKernelGGL((qb_apply<1, false>), QA_ARGS);
#undef QA_ARGS
    launch_select(c, q, w, at, vn1, diag, st);
    LRA_HIP(hipGetLastError());
  }
  return LRA_OK;
}

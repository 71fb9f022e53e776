// snorm.hip -- spectral norm by power iteration (snorm / snormdiff, src/snorm.jl:14-53).
//
// The reference iterates xn <- A'(A xn) (A itself when Hermitian) with s = sqrt(|xn|) and
// stops when |s - t| <= max(atol, t*rtol) or after snorm_niter steps (LRAOptions default 32).
// Each step is two HBM-bound matrix-vector products; they run as GEMV kernels that read A
// once per product.  snormdiff(A, F) applies A - F matrix-free (src/linop.jl:155-187); for an
// ID F = A[:,sk] [I T] P', (A - F) x = A x - A[:,sk] (x[sk] + T x[rd]) and
// (A - F)' y = A' y - P [I T]' A[:,sk]' y, each with a single product with A (op_apply).
#include "lra_internal.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

namespace {

// State of a power iteration, kept on the device: the kernels of a step return at once when
// `done` is set, so the host enqueues several steps before it reads the state.
struct PowerState {
  double s, t, inv;  // estimate, previous estimate, 1 / |x|
  int niter, done;
};

constexpr int GV_ROWS = 512;  // rows of a gemv_n block: two per thread

typedef double d2v __attribute__((ext_vector_type(2)));

// part[c][i] = sum_{j in chunk c} A[i, j] x[cols ? cols[j] - 1 : j].  Bound by reading A: 16-byte
// loads, eight columns in flight per thread (64 KB per CU at eight waves), x from LDS.
// 8192 x 8192: 537 MB in 100 us (5.4 TB/s); one row per thread and one column at a time
// took 150.
template <bool VEC>
__global__ __launch_bounds__(256) void gemv_n_kernel(i64 m, i64 n, const double* __restrict__ A,
                                                     i64 lda, const i64* __restrict__ cols,
                                                     const double* __restrict__ x, i64 chunk,
                                                     double* __restrict__ part,
                                                     const PowerState* st) {
  if (st->done) return;
  constexpr int UN = 8, XT = 512;
  __shared__ double sx[XT];
  const i64 i = (i64)blockIdx.x * GV_ROWS + (VEC ? 2 * threadIdx.x : threadIdx.x);
  const i64 i1 = VEC ? i + 1 : i + 256;
  // rows past the end are read from the last row (pair) and not stored; VEC: m is even
  const i64 q = VEC ? std::min<i64>(i, m - 2) : std::min<i64>(i, m - 1);
  const i64 q1 = VEC ? q + 1 : std::min<i64>(i1, m - 1);
  const i64 j0 = (i64)blockIdx.y * chunk, j1 = std::min<i64>(n, j0 + chunk);
  double a0 = 0.0, a1 = 0.0;
  for (i64 jb = j0; jb < j1; jb += XT) {
    const int nj = (int)std::min<i64>(j1 - jb, XT);
    __syncthreads();
    for (int j = threadIdx.x; j < nj; j += 256) sx[j] = x[cols ? cols[jb + j] - 1 : jb + j];
    __syncthreads();
    const double* a = A + jb * lda;
    int j = 0;
    for (; j + UN <= nj; j += UN) {
      d2v v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        if constexpr (VEC) v[u] = *reinterpret_cast<const d2v*>(a + (i64)(j + u) * lda + q);
        else v[u] = d2v{a[(i64)(j + u) * lda + q], a[(i64)(j + u) * lda + q1]};
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        a0 += v[u].x * sx[j + u];
        a1 += v[u].y * sx[j + u];
      }
    }
    for (; j < nj; ++j) {
      a0 += a[(i64)j * lda + q] * sx[j];
      a1 += a[(i64)j * lda + q1] * sx[j];
    }
  }
  double* p = part + (i64)blockIdx.y * m;
  if (i < m) p[i] = a0;
  if (i1 < m) p[i1] = a1;
}

// y[rows ? rows[i] - 1 : i] = alpha sum_c part[c][i] + beta y[..]: 64 rows per block, each wave
// a quarter of the chunks (fixed order)
__global__ __launch_bounds__(256) void sum_partials_kernel(i64 m, int nchunks,
                                                           const double* __restrict__ part,
                                                           double alpha, double* y, double beta,
                                                           const i64* __restrict__ rows,
                                                           const PowerState* st) {
  if (st->done) return;
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const i64 i = (i64)blockIdx.x * 64 + lane;
  const int per = (nchunks + 3) / 4, c0 = w * per, c1 = min(nchunks, c0 + per);
  double s = 0.0;
  if (i < m) {
#pragma unroll 8
    for (int c = c0; c < c1; ++c) s += part[(i64)c * m + i];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w != 0 || i >= m) return;
  s = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
  double* o = y + (rows ? rows[i] - 1 : i);
  *o = beta == 0.0 ? alpha * s : alpha * s + beta * *o;
}

// y[idx ? idx[j] - 1 : j] = alpha A[:, j]' x + beta y[..], WPC waves on a column (a block each
// for WPC = 4), 16-byte loads (VEC).  Bound by reading A; x comes from L2 with every column and
// does not show: 8192 x 8192 takes 90 us (6.0 TB/s, what a large read reaches) with a block per
// column, 93 with a wave, and 99 / 144 / 230 with 2 / 4 / 8 columns per wave sharing x, which
// leaves fewer waves in flight.  8-byte loads, a wave per column: 143.
template <int WPC, bool VEC>
__global__ __launch_bounds__(256) void gemv_t_kernel(i64 m, i64 n, const double* __restrict__ A,
                                                     i64 lda, const i64* __restrict__ idx,
                                                     const double* __restrict__ x, double alpha,
                                                     double* y, double beta,
                                                     const PowerState* st) {
  if (st->done) return;
  static_assert(WPC == 1 || WPC == 4, "a wave or a block per column");
  constexpr int W = 64 * WPC;  // threads on a column
  __shared__ double red[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const i64 j = WPC == 4 ? (i64)blockIdx.x : (i64)blockIdx.x * 4 + w;
  if (WPC == 1 && j >= n) return;
  const int t = WPC == 4 ? (int)threadIdx.x : lane;
  const double* a = A + j * lda;
  double s = 0.0;
  if constexpr (VEC) {
#pragma unroll 4
    for (i64 i = 2 * t; i + 1 < m; i += 2 * W) {
      const d2v xv = *reinterpret_cast<const d2v*>(x + i);
      const d2v v = *reinterpret_cast<const d2v*>(a + i);
      s += v.x * xv.x;
      s += v.y * xv.y;
    }
    if ((m & 1) && t == 0) s += a[m - 1] * x[m - 1];
  } else {
#pragma unroll 4
    for (i64 i = t; i < m; i += W) s += a[i] * x[i];
  }
  s = lra_wave_sum(s);
  if constexpr (WPC == 4) {
    if (lane == 0) red[w] = s;
    __syncthreads();
    s = (red[0] + red[1]) + (red[2] + red[3]);
  }
  if (t != 0) return;
  double* o = y + (idx ? idx[j] - 1 : j);
  *o = beta == 0.0 ? alpha * s : alpha * s + beta * *o;
}

// w[r] = y[sk[r] - 1], and that entry of y cleared
__global__ void take_rows_kernel(i64 k, const i64* __restrict__ sk, double* y, double* w,
                                 const PowerState* st) {
  if (st->done) return;
  for (i64 r = blockIdx.x * (i64)blockDim.x + threadIdx.x; r < k; r += (i64)gridDim.x * blockDim.x) {
    w[r] = y[sk[r] - 1];
    y[sk[r] - 1] = 0.0;
  }
}

// One step's end (one block): |x|, the new estimate and the stop test (src/snorm.jl:35-43); x is
// scaled to unit length when it fits the block's registers (else scale_kernel follows).
// first: only the length of the start vector.
constexpr int NS_T = 1024, NS_R = 16;
__global__ __launch_bounds__(NS_T) void norm_step_kernel(i64 n, double* x, int first, int isherm,
                                                         double atol, double rtol, i64 maxit,
                                                         PowerState* st) {
  if (!first && st->done) return;
  __shared__ double red[NS_T / 64];
  const bool held = n <= NS_T * NS_R;
  double v[NS_R];
  double s = 0.0;
  if (held) {
#pragma unroll
    for (int r = 0; r < NS_R; ++r) {
      const i64 i = threadIdx.x + (i64)r * NS_T;
      v[r] = i < n ? x[i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < NS_R; ++r) s += v[r] * v[r];
  } else {
#pragma unroll 8
    for (i64 i = threadIdx.x; i < n; i += NS_T) s += x[i] * x[i];
  }
  s = lra_wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  double tot = 0.0;
#pragma unroll
  for (int w = 0; w < NS_T / 64; ++w) tot += red[w];
  const double nrm = sqrt(tot), inv = 1.0 / nrm;
  if (held) {
#pragma unroll
    for (int r = 0; r < NS_R; ++r) {
      const i64 i = threadIdx.x + (i64)r * NS_T;
      if (i < n) x[i] = v[r] * inv;
    }
  }
  if (threadIdx.x == 0) {
    st->inv = inv;
    if (first) {
      st->s = 1.0;
      st->t = 0.0;
      st->niter = 0;
      st->done = 0;
    } else {
      const double t = st->s, e = isherm ? nrm : sqrt(nrm);
      st->t = t;
      st->s = e;
      const int it = ++st->niter;
      const bool go = e > 0 && fabs(e - t) > fmax(atol, t * rtol);
      if (!go || it == maxit) st->done = 1;
    }
  }
}

__global__ void scale_kernel(i64 n, double* x, const PowerState* st) {
  if (st->done) return;
  const double inv = st->inv;
  for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
    x[i] *= inv;
}

inline int blocks_for(i64 n) { return (int)std::min<i64>(std::max<i64>((n + 255) / 256, 1), 4096); }

// column chunks of gemv_n for an m x n product (the partial sums are chunks x m): about four
// blocks per CU, chunks of at least 16 columns; `most` doubles of partial sums at the most
i64 gemv_chunks(const lra_ctx* c, i64 m, i64 n, size_t most, i64* chunk) {
  const i64 rt = (m + GV_ROWS - 1) / GV_ROWS;
  i64 nch = std::max<i64>(1, std::min<i64>((n + 15) / 16, (4ll * c->num_cu + rt - 1) / rt));
  nch = std::max<i64>(1, std::min<i64>(nch, (i64)(most / (size_t)std::max<i64>(m, 1))));
  *chunk = std::max<i64>(1, (n + nch - 1) / nch);
  return n > 0 ? (n + *chunk - 1) / *chunk : 1;
}

// The number of chunks of at least 256 columns for about four blocks of 256 rows per CU: the partial
// sums that a caller with little memory has room for (lra_snormdiff_id_noalloc's array, a context
// with a scratch limit).
i64 least_chunks(const lra_ctx* c, i64 m, i64 n) {
  const i64 rt = std::max<i64>(1, (m + 255) / 256);
  return std::max<i64>(1, std::min<i64>((n + 255) / 256, (4ll * c->num_cu + rt - 1) / rt));
}

// whether rows (pairs of doubles) of A and x can be read 16 bytes at a time
bool pairs_ok(const double* A, i64 lda, const double* x, i64 m) {
  return m >= 2 && lda % 2 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)x & 15) == 0;
}

struct Gemv {
  lra_ctx* c;
  const PowerState* st;
  double* part = nullptr;  // caller's partial sums, of `most` doubles (else a workspace slot)
  size_t most = ~(size_t)0;

  // y[rows] = alpha A x[cols] + beta y[rows]  (rows, cols optional, 1-based)
  int n(i64 m, i64 nn, const double* A, i64 lda, const i64* cols, const double* x, double alpha,
        double* y, double beta, const i64* rows = nullptr) const {
    if (m <= 0) return LRA_OK;
    i64 chunk = 0;
    i64 nch = gemv_chunks(c, m, nn, most, &chunk);
    double* p = part;
    if (!p) {
      int rc = lra_wsT(c, WS_X0, (size_t)nch * m, &p);
      if (rc == LRA_E_ALLOC && nch > 1) {  // a budget without room for them: one range
        nch = 1;
        chunk = nn;
        rc = lra_wsT(c, WS_X0, (size_t)m, &p);
      }
      LRA_CHECK(rc);
    }
    if (nn > 0) {
      const dim3 grid((unsigned)((m + GV_ROWS - 1) / GV_ROWS), (unsigned)nch);
      if (m % 2 == 0 && pairs_ok(A, lda, A, m))
        hipLaunchKernelGGL(gemv_n_kernel<true>, grid, dim3(256), 0, c->stream, m, nn, A, lda,
                           cols, x, chunk, p, st);
      else
        hipLaunchKernelGGL(gemv_n_kernel<false>, grid, dim3(256), 0, c->stream, m, nn, A, lda,
                           cols, x, chunk, p, st);
    }
    hipLaunchKernelGGL(sum_partials_kernel, dim3((unsigned)((m + 63) / 64)), dim3(256), 0,
                       c->stream, m, nn > 0 ? (int)nch : 0, p, alpha, y, beta, rows, st);
    LRA_HIP(hipGetLastError());
    return LRA_OK;
  }

  // y[idx] = alpha A' x + beta y[idx]  (idx optional, 1-based)
  int t(i64 m, i64 nn, const double* A, i64 lda, const i64* idx, const double* x, double alpha,
        double* y, double beta) const {
    if (nn <= 0) return LRA_OK;
    const bool vec = pairs_ok(A, lda, x, m);
    // a column of 436 rows does not fill a block: 8.8 us for T (436 x 7756) with a wave per
    // column, 9.4 with a block; from 1024 rows on the block
    const bool block = m >= 1024;
    const dim3 grid((unsigned)(block ? nn : (nn + 3) / 4));
#define GT_ARGS grid, dim3(256), 0, c->stream, m, nn, A, lda, idx, x, alpha, y, beta, st
    if (block && vec) hipLaunchKernelGGL((gemv_t_kernel<4, true>), GT_ARGS);
    else if (block) hipLaunchKernelGGL((gemv_t_kernel<4, false>), GT_ARGS);
    else if (vec) hipLaunchKernelGGL((gemv_t_kernel<1, true>), GT_ARGS);
    else hipLaunchKernelGGL((gemv_t_kernel<1, false>), GT_ARGS);
#undef GT_ARGS
    LRA_HIP(hipGetLastError());
    return LRA_OK;
  }
};

struct Op {
  // (A - F) where F is an ID of A (k > 0) or nothing (k < 0)
  i64 m, n;
  const double* A;
  i64 lda;
  i64 k;
  const i64* sk;
  const i64* rd;
  const double* T;
  i64 ldt;
  const double* B;  // second dense operand (snormdiff of two matrices) or nullptr
  i64 ldb;
  lra_apply_fn apply = nullptr;  // matrix-free operator (replaces A when set)
  void* user = nullptr;
  double* part = nullptr;  // partial-sum buffer of the GEMVs (else a workspace slot)
  size_t most = ~(size_t)0;  // its doubles
};

int op_callback(lra_ctx* c, const Op& o, int trans, const double* x, i64 ldx, double* y, i64 ldy) {
  const int st = o.apply(o.user, trans, 1, x, std::max<i64>(ldx, 1), y, std::max<i64>(ldy, 1),
                         (void*)c->stream);
  if (st != 0) { lra_set_error("operator apply returned %d", st); return LRA_E_STATE; }
  return LRA_OK;
}

// y = (A - F) x.  F takes A's own skeleton columns, so the two products with A are one:
// (A - F) x = A x - A[:, sk] (x[sk] + T x[rd]) = A x' with x'[rd] = x[rd], x'[sk] = -T x[rd].
// x is overwritten by x'.
int op_apply(lra_ctx* c, const Op& o, double* x, double* y, const PowerState* st) {
  if (o.apply) return op_callback(c, o, 0, x, o.n, y, o.m);
  const Gemv g{c, st, o.part, o.most};
  const i64 seg = (i64)std::min<size_t>((size_t)std::max<i64>(o.k, 1), o.most);  // rows of T
  for (i64 r = 0; r < o.k; r += seg)
    LRA_CHECK(g.n(std::min(seg, o.k - r), o.n - o.k, o.T + r, o.ldt, o.rd, x, -1.0, x, 0.0,
                  o.sk + r));
  LRA_CHECK(g.n(o.m, o.n, o.A, o.lda, nullptr, x, 1.0, y, 0.0));
  if (o.B) LRA_CHECK(g.n(o.m, o.n, o.B, o.ldb, nullptr, x, -1.0, y, 1.0));
  return LRA_OK;
}

// y = (A - F)' x.  A[:, sk]' x is the entries sk of A' x, so with w = (A' x)[sk] the rest is
// y[sk] = 0, y[rd] = (A' x)[rd] - T' w.
int op_apply_t(lra_ctx* c, const Op& o, const double* x, double* y, double* wk,
               const PowerState* st) {
  if (o.apply) return op_callback(c, o, 1, x, o.m, y, o.n);
  const Gemv g{c, st, o.part, o.most};
  LRA_CHECK(g.t(o.m, o.n, o.A, o.lda, nullptr, x, 1.0, y, 0.0));
  if (o.B) LRA_CHECK(g.t(o.m, o.n, o.B, o.ldb, nullptr, x, -1.0, y, 1.0));
  if (o.k > 0) {
    hipLaunchKernelGGL(take_rows_kernel, dim3(blocks_for(o.k)), dim3(256), 0, c->stream, o.k, o.sk,
                       y, wk, st);
    LRA_HIP(hipGetLastError());
    LRA_CHECK(g.t(o.k, o.n - o.k, o.T, o.ldt, o.rd, wk, -1.0, y, 1.0));
  }
  return LRA_OK;
}

// Vectors of the power iteration: xn (n), xm (m), wk (max(k,1) + 64; its tail holds the state).
struct PowerBufs {
  double *xn, *xm, *wk;
};

// power iteration loop of snorm (src/snorm.jl:14-45); buffers from the workspace unless given.
// The estimate and the stop test are on the device: the host enqueues four steps, then eight
// at a time, and reads the state after each batch (steps after the stop return at once).  A
// caller's operator is applied exactly as often as the reference applies it: one step at a time.
int power_iteration(lra_ctx* c, const Op& op, int isherm, const lra_opts* opts, const double* x0,
                    double* result, const PowerBufs* given = nullptr) {
  Op o = op;
  const i64 m = o.m, n = o.n;
  // (what a limited context gives to partial sums it holds from here on: more of them than these
  // would take the room of the calls that follow)
  if (!given && c->hbm_budget != 0) o.most = (size_t)std::max<i64>(1, least_chunks(c, m, n) * m);
  double *xn = nullptr, *xm = nullptr, *wk = nullptr;
  if (given) {
    xn = given->xn; xm = given->xm; wk = given->wk;
  } else {
    LRA_CHECK(lra_wsT(c, WS_QR0, (size_t)std::max<i64>(n, 1), &xn));
    LRA_CHECK(lra_wsT(c, WS_QR1, (size_t)std::max<i64>(m, 1), &xm));
    LRA_CHECK(lra_wsT(c, WS_QR2, (size_t)std::max<i64>(std::max<i64>(o.k, 1), 1) + 64, &wk));
  }
  PowerState* st = reinterpret_cast<PowerState*>(wk + std::max<i64>(o.k, 1));
  *result = 1.0;
  if (opts->snorm_niter == 0 || !(1.0 > opts->atol)) return LRA_OK;
  if (x0) LRA_HIP(hipMemcpyAsync(xn, x0, sizeof(double) * n, hipMemcpyDeviceToDevice, c->stream));
  else LRA_CHECK(lra_launch_gaussian_fill(c->stream, opts->seed, 0x5A0A5A0Aull, n, 1, xn, n));
  auto norm_step = [&](double* x, int first) -> int {
    hipLaunchKernelGGL(norm_step_kernel, dim3(1), dim3(NS_T), 0, c->stream, n, x, first, isherm,
                       opts->atol, opts->rtol, (i64)opts->snorm_niter, st);
    if (n > NS_T * NS_R)
      hipLaunchKernelGGL(scale_kernel, dim3(blocks_for(n)), dim3(256), 0, c->stream, n, x, st);
    LRA_HIP(hipGetLastError());
    return LRA_OK;
  };
  LRA_CHECK(norm_step(xn, 1));
  PowerState* hs = (PowerState*)c->host_pinned;
  i64 left = opts->snorm_niter;  // (negative: until it converges)
  for (int batch = o.apply ? 1 : 4;; batch = o.apply ? 1 : 8) {
    for (int b = 0; b < batch && left != 0; ++b, --left) {
      LRA_CHECK(op_apply(c, o, xn, xm, st));
      if (isherm) std::swap(xn, xm);
      else LRA_CHECK(op_apply_t(c, o, xm, xn, wk, st));
      LRA_CHECK(norm_step(xn, 0));
    }
    LRA_HIP(hipMemcpyAsync(hs, st, sizeof(PowerState), hipMemcpyDeviceToHost, c->stream));
    LRA_HIP(hipStreamSynchronize(c->stream));
    if (hs->done) break;
  }
  *result = hs->s;
  return LRA_OK;
}

}  // namespace

extern "C" int lra_snorm(lra_ctx* c, int64_t m, int64_t n, const double* A, int64_t lda,
                         int isherm, const lra_opts* opts, const double* x0, double* result) {
  LRA_ARG(c != nullptr, 1);
  LRA_ARG(m >= 0, 2);
  LRA_ARG(n >= 0, 3);
  LRA_ARG(lda >= std::max<int64_t>(1, m), 5);
  LRA_ARG(!isherm || m == n, 6);
  LRA_ARG(opts != nullptr, 7);
  LRA_ARG(result != nullptr, 9);
  Op o{m, n, A, lda, -1, nullptr, nullptr, nullptr, 0, nullptr, 0};
  return power_iteration(c, o, isherm, opts, x0, result);
}

extern "C" int lra_snormdiff(lra_ctx* c, int64_t m, int64_t n, const double* A, int64_t lda,
                             const double* B, int64_t ldb, int isherm, const lra_opts* opts,
                             const double* x0, double* result) {
  LRA_ARG(c != nullptr, 1);
  LRA_ARG(m >= 0, 2);
  LRA_ARG(n >= 0, 3);
  LRA_ARG(lda >= std::max<int64_t>(1, m), 5);
  LRA_ARG(B != nullptr, 6);
  LRA_ARG(ldb >= std::max<int64_t>(1, m), 7);
  LRA_ARG(opts != nullptr, 9);
  LRA_ARG(result != nullptr, 11);
  Op o{m, n, A, lda, -1, nullptr, nullptr, nullptr, 0, B, ldb};
  return power_iteration(c, o, isherm, opts, x0, result);
}

extern "C" int lra_snormdiff_id(lra_ctx* c, int64_t m, int64_t n, const double* A, int64_t lda,
                                int64_t k, const int64_t* sk, const int64_t* rd, const double* T,
                                int64_t ldt, const lra_opts* opts, const double* x0,
                                double* result) {
  LRA_ARG(c != nullptr, 1);
  LRA_ARG(m >= 0, 2);
  LRA_ARG(n >= 0, 3);
  LRA_ARG(lda >= std::max<int64_t>(1, m), 5);
  LRA_ARG(k >= 0 && k <= n, 6);
  LRA_ARG(ldt >= std::max<int64_t>(1, k), 10);
  LRA_ARG(opts != nullptr, 11);
  LRA_ARG(result != nullptr, 13);
  Op o{m, n, A, lda, k, sk, rd, T, ldt, nullptr, 0};
  if (k == 0) o.k = -1;
  return power_iteration(c, o, 0, opts, x0, result);
}

// snorm of a matrix-free operator (snorm(L::LinearOperator), src/snorm.jl:14-45): the power
// iteration applies the caller's L and L' to one vector per step.
extern "C" int lra_snorm_op(lra_ctx* c, int64_t m, int64_t n, lra_apply_fn apply, void* user,
                            int isherm, const lra_opts* opts, const double* x0, double* result) {
  LRA_ARG(c != nullptr, 1);
  LRA_ARG(m >= 0, 2);
  LRA_ARG(n >= 0, 3);
  LRA_ARG(apply != nullptr, 4);
  LRA_ARG(!isherm || m == n, 6);
  LRA_ARG(opts != nullptr, 7);
  LRA_ARG(result != nullptr, 9);
  Op o{m, n, nullptr, 1, -1, nullptr, nullptr, nullptr, 0, nullptr, 0};
  o.apply = apply;
  o.user = user;
  return power_iteration(c, o, isherm, opts, x0, result);
}

// ---------------------------------------------------------------------------------------
// Allocation-free variant of lra_snormdiff_id.  All of its device memory beyond the caller's
// inputs is `scratch`, a file-scope device array of kScratchDoubles doubles (32 MiB) that
// every GPU the library runs on holds until the process ends.  On the host the array's name
// is only a stand-in: its device address is fetched per device with hipGetSymbolAddress on the
// first call on that device (with the device current) and kept in g_scratch; only that
// address is handed to kernels.  Calls on one GPU share its array (the last call's contents
// stay behind; every element a call reads it has written first, so nothing is cleared), and
// calls that overlap on one GPU race.

static constexpr size_t kScratchDoubles = (size_t)4 << 20;
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
std::mutex g_scratch_mu;
double* g_scratch[64] = {};

int scratch_on(int device, double** out) {
  if (device < 0 || device >= 64) {
    lra_set_error("scratch: device %d out of range", device);
    return LRA_E_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[device]) {
    LRA_HIP(hipSetDevice(device));
    void* p = nullptr;
    LRA_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[device] = static_cast<double*>(p);
  }
  *out = g_scratch[device];
  return LRA_OK;
}
}  // namespace

extern "C" int lra_snormdiff_id_noalloc(lra_ctx* c, int64_t m, int64_t n, const double* A,
                                        int64_t lda, int64_t k, const int64_t* sk,
                                        const int64_t* rd, const double* T, int64_t ldt,
                                        const lra_opts* opts, const double* x0,
                                        double* result) {
  LRA_ARG(c != nullptr, 1);
  LRA_ARG(m >= 0, 2);
  LRA_ARG(n >= 0, 3);
  LRA_ARG(lda >= std::max<int64_t>(1, m), 5);
  LRA_ARG(k >= 0 && k <= n, 6);
  LRA_ARG(ldt >= std::max<int64_t>(1, k), 10);
  LRA_ARG(opts != nullptr, 11);
  LRA_ARG(result != nullptr, 13);
  // scratch layout: xn (n) | xm (m) | wk (max(k,1) + 64) | GEMV partial sums, with what is left
  // (at least the sums of `least_chunks`)
  const i64 nparts = least_chunks(c, m, n);
  const size_t head = (size_t)std::max<i64>(n, 1) + (size_t)std::max<i64>(m, 1) +
                      (size_t)std::max<i64>(k, 1) + 64;
  const size_t need = head + (size_t)nparts * (size_t)m;
  if (need > kScratchDoubles) {
    lra_set_error("snormdiff_id_noalloc: %zu doubles of scratch needed for m=%lld n=%lld "
                  "k=%lld, the maximum is %zu (use lra_snormdiff_id)", need, (long long)m,
                  (long long)n, (long long)k, kScratchDoubles);
    return LRA_E_UNSUPPORTED;
  }
  double* base = nullptr;
  LRA_CHECK(scratch_on(c->device, &base));
  LRA_HIP(hipSetDevice(c->device));
  PowerBufs b;
  b.xn = base;
  // (16-byte aligned vectors: two of the 64 spare doubles, the state takes five)
  b.xm = b.xn + (std::max<i64>(n, 1) + 1) / 2 * 2;
  b.wk = b.xm + (std::max<i64>(m, 1) + 1) / 2 * 2;
  Op o{m, n, A, lda, k, sk, rd, T, ldt, nullptr, 0};
  o.part = base + head;
  o.most = std::max<size_t>(kScratchDoubles - head, 1);
  if (k == 0) o.k = -1;
  return power_iteration(c, o, 0, opts, x0, result, &b);
}

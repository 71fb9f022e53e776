// lra_qg.h -- state shared by the HBM pivoted-QR kernels (qrcp_global.hip: one launch per step;
// qrcp_block.hip: blocks of steps).
#pragma once
#include "lra_internal.h"

struct FState {
  int j0, jb, done, k, early;  // dlaqps block start and length, stop state, rank
  int sprev;       // last single step whose pivot column is still to be rewritten, or -1
  int s, b;        // next step; steps of the block just applied (their bookkeeping is pending)
  int ncand;       // candidates of the next block (0: the block cannot run)
  unsigned mask;   // bit t: a column norm was recomputed after step s + t
  double ptol;
  double tau;      // largest column norm outside the candidates
};

// Workspace of the block steps: candidates, Gram matrix, reflectors in tiles of 16 rows (each
// column-major, 16 columns), the block's tau.
struct QbWork {
  int* cand;    // storage columns (QB_C), then positions (QB_C), then the block's swaps (16)
  double* G;    // QB_C x QB_C
  double* V;    // (m rounded up to 16) x 16
  double* T;    // tau of the block (16)
};
constexpr int QB_C = 128, QB_B = 16;
inline size_t lra_qb_doubles(int m) {
  return (size_t)QB_C + 16 + (size_t)QB_C * QB_C + ((size_t)m + 31) / 16 * 256 + 256;
}
QbWork lra_qb_work(double* w, int m);

// Steps a block of that many rows holds: the panel keeps its columns in the registers of one
// workgroup, at most 36 doubles a thread.
inline int lra_qb_cap(int rows) { return rows <= 2048 ? 16 : rows <= 3072 ? 12 : rows <= 4096 ? 8 : 4; }

// Selects the candidates of the first block.
int lra_qb_start(lra_ctx* c, const QrcpCall& q, const QbWork& w, const int* at, double* vn1,
                 const double* diag, FState* st);
// `count` blocks of at most QB_B steps; `s` is a step no later than the state's.
int lra_qb_blocks(lra_ctx* c, const QrcpCall& q, const QbWork& w, int* at, double* vn1,
                  double* vn2, double* diag, FState* st, int s, int count);
// The pivot of the state's step moved to its position (before single steps).
int lra_qb_pick(lra_ctx* c, const QbWork& w, int* at, FState* st);

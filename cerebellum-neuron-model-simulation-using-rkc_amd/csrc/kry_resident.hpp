// A whole CG / BiCG solve of the CN and BE paths in one kernel.
//
// The reference's solve is 100 iterations of two dot products each, most of
// them far from convergence.  As two launches per iteration whose last block
// reduced every block's partial sum, an iteration of 102400 compartments took
// 29 us: the release of each block's partial writes back its XCD's L2, and the
// 100 iterations are a serial chain of 200 such launches.  Here a workgroup
// keeps its rows (whole 256-row chunks) for the whole solve, x, r and A p in
// registers, p and its part of the matrix in LDS, and the dot products are
// grid_sum exchanges.  Neighbours beyond the workgroup's rows are ghosts: r of
// the rows that others need is posted with each update, and every workgroup
// advances its ghosts' p by the recurrence its owner uses.  Products, row sums
// and dot products are those of k_kry_a / k_kry_b in the same order, so the
// iterates are the same bit for bit.
// Measured, calls of Population.run (us): 64 Purkinje cells (102400 rows, 200
// workgroups), 10 solves of 100 CG iterations, 29430 -> 10620, 10.2 an
// iteration, nearly all of it the two exchanges; 1024 olive cells (3072 rows,
// 6 workgroups), 40 BiCG solves, 13440 -> 3470 (one workgroup of 256 threads
// with its vectors in global memory before).
#pragma once
#include <hip/hip_runtime.h>

#include "grid_mail.hpp"

namespace cbrkc {

struct KryArgs {
  int nc, nch, rb;                       // rows, chunks, rows of a workgroup
  int nnz_max, ghost_max;                // LDS sizes
  // local rows: workgroup w's start at lrow[w (rb + 1)], entries with the
  // diagonal in column order, columns local (ghosts from rb on), dpos the local
  // diagonal entry; the transpose likewise (BiCG)
  const unsigned short *lrow, *lcol, *ldpos;
  const double *lval;
  const int *lnz0;
  const unsigned short *trow, *tcol, *tdpos;
  const double *tval;
  const int *imp0, *imp;                 // ghosts fetched (null: none), their rows
  const int *exp0;                       // rows posted, sorted by the thread that holds them:
  const int *exp_t0;                     // thread t of workgroup w posts [exp_t0[w NT + t], exp_t0[w NT + t + 1])
  const int *exp_row, *exp_slot;
  double *ghost;                         // [3][2][nslot]: r, and BiCG's shadow residual
  int nslot;
  double *parts;                         // [3][nch]
  unsigned *q;                           // number (modulo 3) of the next sum; nonzero once a wait gave up
  int *late;                             // the same in mapped host memory
  unsigned long long wait;               // the limit of a wait (grid_mail.hpp)
  const double *diag, *b;
  double *v;
  int *flag, f_done, f_iters, f_total;
};

template <int NT, int K, bool BICG>
__global__ void __launch_bounds__(NT) k_kry_resident(KryArgs A) {
  extern __shared__ double sm[];
  __shared__ int s_late;
  const int tid = threadIdx.x, w = blockIdx.x, r0 = w * A.rb, R = min(A.rb, A.nc - r0), ps = A.rb + A.ghost_max;
  double *P = sm, *PS = P + ps, *T = BICG ? PS + ps : PS, *part = T + A.rb, *LV = part + A.nch + 8;
  double *TV = LV + A.nnz_max;
  unsigned short *LR = (unsigned short *)(BICG ? TV + A.nnz_max : TV), *LC = LR + A.rb + 1;
  unsigned short *TR = LC + A.nnz_max, *TC = TR + A.rb + 1;
  SumPlan S;
  S.set(A.nc, r0, r0 + R);
  Wait W{A.wait, &s_late, 0};
  bool late = false;
  unsigned q = A.q[0];
  // a solve before this one ended with its mailboxes half read: those already
  // queued after it fall through
  if (A.q[1]) return;
  if (tid == 0) s_late = 0;
  const int z0 = A.lnz0[w], nz = A.lnz0[w + 1] - z0;
  for (int k = tid; k < nz; k += NT) {
    LV[k] = A.lval[z0 + k];
    LC[k] = A.lcol[z0 + k];
    if (BICG) {
      TV[k] = A.tval[z0 + k];
      TC[k] = A.tcol[z0 + k];
    }
  }
  for (int i = tid; i <= R; i += NT) {
    LR[i] = A.lrow[(size_t)w * (A.rb + 1) + i];
    if (BICG) TR[i] = A.trow[(size_t)w * (A.rb + 1) + i];
  }
  const int g0 = A.imp0 ? A.imp0[w] : 0, ng = A.imp0 ? A.imp0[w + 1] - g0 : 0;
  const int e0 = A.imp0 ? A.exp0[w] : 0, ne = A.imp0 ? A.exp0[w + 1] - e0 : 0;
  const int t0 = A.imp0 ? A.exp_t0[w * NT + tid] : 0, t1 = A.imp0 ? A.exp_t0[w * NT + tid + 1] : 0;
  const int row0 = t0 < t1 ? A.exp_row[t0] : 0, slot0 = t0 < t1 ? A.exp_slot[t0] : 0;
  {   // what the last solve posted with its last update and nobody read
    double *old = A.ghost + (size_t)(q == 0 ? 2 : q - 1) * 2 * A.nslot;
    for (int k = tid; k < ne; k += NT) {
      mail_clear(old + A.exp_slot[e0 + k]);
      if (BICG) mail_clear(old + A.nslot + A.exp_slot[e0 + k]);
    }
  }
  __syncthreads();
  double x[K], r[K], ap[K], rs[K], atp[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int i = tid + k * NT;
    x[k] = r[k] = rs[k] = ap[k] = atp[k] = 0.0;
    if (i < R) {
      const double bi = A.b[r0 + i], di = A.diag[r0 + i];
      x[k] = 0.0 * A.v[r0 + i];   // cublasDscal by 0 (solve_cnm.cu:65)
      r[k] = rs[k] = bi;
      P[i] = bi;
      LV[A.ldpos[r0 + i]] = di;
      if (BICG) {
        PS[i] = bi;
        TV[A.tdpos[r0 + i]] = di;
      }
      T[i] = bi * bi;
    }
  }
  for (int g = tid; g < ng; g += NT) {
    const double bi = A.b[A.imp[g0 + g]];
    P[A.rb + g] = bi;
    if (BICG) PS[A.rb + g] = bi;
  }
  auto sum = [&]() { return grid_sum<NT>(S, T, part, (double *)nullptr, A.parts, q, W, late); };
  const double bnorm = sum();
  double rr = bnorm, beta = 0.0;
  int iters = 0, done = 0;
  for (int k = 0; k < 100 && !done && !late; k++) {
    if (k > 0) {   // p = beta p + r, ghosts included (posted before the last sum)
      const double *gq = A.ghost + (size_t)(q == 0 ? 2 : q - 1) * 2 * A.nslot;
#pragma unroll
      for (int j = 0; j < K; j++) {
        const int i = tid + j * NT;
        if (i < R) {
          P[i] = beta * P[i] + r[j];
          if (BICG) PS[i] = beta * PS[i] + rs[j];
        }
      }
      for (int g = tid; g < ng; g += NT) {
        P[A.rb + g] = beta * P[A.rb + g] + mail_get(gq + g0 + g, W);
        if (BICG) PS[A.rb + g] = beta * PS[A.rb + g] + mail_get(gq + A.nslot + g0 + g, W);
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int i = tid + j * NT;
      if (i < R) {
        double s = 0.0;
        const int e = LR[i + 1];
        for (int n = LR[i]; n < e; n++) s += LV[n] * P[LC[n]];
        ap[j] = s;
        if (BICG) {
          double st = 0.0;
          const int te = TR[i + 1];
          for (int n = TR[i]; n < te; n++) st += TV[n] * PS[TC[n]];
          atp[j] = st;
          T[i] = PS[i] * s;
        } else {
          T[i] = P[i] * s;
        }
      }
    }
    const double alpha = rr / sum(), nalpha = -1.0 * alpha;
    // the ghosts of the last update have been read by everybody
    if (ne > 0 && k > 0) {
      double *old = A.ghost + (size_t)(q == 2 ? 0 : q + 1) * 2 * A.nslot;
      for (int n = tid; n < ne; n += NT) {
        mail_clear(old + A.exp_slot[e0 + n]);
        if (BICG) mail_clear(old + A.nslot + A.exp_slot[e0 + n]);
      }
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int i = tid + j * NT;
      if (i < R) {
        x[j] = alpha * P[i] + x[j];
        r[j] = nalpha * ap[j] + r[j];
        if (BICG) {
          rs[j] = nalpha * atp[j] + rs[j];
          T[i] = r[j] * rs[j];
        } else {
          T[i] = r[j] * r[j];
        }
      }
    }
    // post what other workgroups need of r: the thread that holds the row
    // (seldom more than one)
    for (int n = t0; n < t1; n++) {
      const int kk = (n == t0 ? row0 : A.exp_row[n]) / NT, slot = n == t0 ? slot0 : A.exp_slot[n];
      double rv = 0.0, rsv = 0.0;
#pragma unroll
      for (int j = 0; j < K; j++)
        if (kk == j) {
          rv = r[j];
          rsv = rs[j];
        }
      double *gq = A.ghost + (size_t)q * 2 * A.nslot;
      mail_put(gq + slot, rv);
      if (BICG) mail_put(gq + A.nslot + slot, rsv);
    }
    const double tot = sum();
    iters = k + 1;
    if (sqrt(tot) <= 1.0e-15 * sqrt(bnorm)) {
      done = 1;
    } else {
      beta = tot / rr;
      rr = tot;
    }
  }
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int i = tid + j * NT;
    if (i < R) A.v[r0 + i] = x[j];
  }
  if (tid == 0 && late) {
    A.q[1] = 1u;
    *A.late = 1;
  }
  if (w == 0 && tid == 0) {
    A.flag[A.f_iters] = iters;
    A.flag[A.f_done] = 1;
    A.flag[A.f_total] += iters;
    *A.q = q;
  }
}

}  // namespace cbrkc

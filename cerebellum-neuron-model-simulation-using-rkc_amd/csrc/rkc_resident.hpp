// The population-global RKC controller and its steps in one kernel: many
// macro steps of rkclow / step / rkcrho (solve_rkc.cu:562-1096) and the ion
// updates between them without the host.
//
// What it replaces took one launch per Chebyshev stage, four more and a read
// back by the host per step attempt: 3-5 us a launch whatever the population
// (two thirds of a small population's time), plus the host's answer.  Here
// every workgroup owns whole cells, keeps their five vectors in LDS and its rows
// of the cable matrix in registers and runs the controller's scalar arithmetic itself
// on the same sums; a stage costs a barrier, a step attempt one exchange of
// the error norm's partial sums.  Cells whose cable matrix couples them
// (gap junctions) also exchange the coupled compartments' values at every
// stage.  The additions of every right-hand side, stage and norm are those of
// the launch-per-stage path in the same order, and what either takes from libm
// the other does too, so the two agree bit for bit.
// Measured, Population.run from the initial state and then on average over the
// eleven calls after it, launch per stage -> this kernel (ms): 64 olive cells, 40
// macro steps, 101 / 15.3 -> 12.0 / 3.1; 256 Golgi cells, 40 steps, 22.7 / 65.9 -> 8.7 /
// 24.8; 16 granule cells, one step, 39.6 / 26.5 -> 10.1 / 6.9; 64 coupled Purkinje
// cells, 8 steps, 9.3 / 2.9 -> 4.6 / 1.5; 9 uncoupled ones 6.5 / 8.1 -> 2.9 / 3.9.
#pragma once
#include <hip/hip_runtime.h>

#include "exp_acc.hpp"
#include "grid_mail.hpp"
#include "philox.hpp"

namespace cbrkc {

// The controller between launches (solve_rkc.cu's others[] and hwork[]), one
// record per population
struct RkcCtl {
  double o[16], hw[8];
  double sum_dt;
  double errold3;             // o[ERROLD]^(1/3)
  double err, h;              // of the step attempt that stopped the kernel (status NONFINITE, ASK_POW)
  long long steps, rejects, stages, rho_iters, ions, macro;
  int last, newspc, jacatt, status;
  unsigned q, ions_q;         // numbers (modulo 3) of the next sum and gap-current exchange
  int ghost_used;             // coupled-value exchanges before the last sum
  int loops;
  int m;                      // stages of the attempt that stopped the kernel (status ASK_STAGE)
  int ghost_now;              // coupled-value exchanges since the last sum
};

// Stage counts up to RES_COEF read their coefficients from the table.  Larger
// ones run the recurrence in the kernel from w1 and mu~_1, whose logarithm and
// hyperbolic functions the host's libm gives: a table up to RES_START stages, and
// beyond it the kernel ends to ask.  (The device's own functions differ in the
// last bit, which a step of 176 stages, taken by Golgi cells as their synaptic
// input sets in, carries to 1e-10 mV.)
constexpr int ASK_POW = 9;     // status: the host has to give the powers of err
constexpr int ASK_STAGE = 10;  // status: the host has to give w1 and mu~_1 for m
constexpr int ASK_DECAY = 11;  // status: the host has to give the synaptic decay of the ion update over sum_dt
constexpr int RES_COEF = 128;
constexpr int RES_START = 4096;
constexpr int RES_COEFS = (RES_COEF + 1) * RES_COEF * 4;   // doubles of the coefficient table
constexpr int ROW_W = 3;            // neighbours of a compartment held in registers (parent and two children)
constexpr int GHOST_STAGES = 136;   // exchanges of coupled values between two sums

struct RkcArgs {
  int n, nc, comp, nblk, cpb;            // cells, rows, rows per cell, workgroups, cells per workgroup
  int ext_max, ghost_max, nch;           // LDS sizes: further entries and ghosts of a workgroup, chunks
  // the rows of the cable matrix without the diagonal, columns local (ghosts from the
  // workgroup's row count on): the first ROW_W entries of row i in lval[k nc + i]
  // and the 16-bit quarters of lcol[i], whose last holds the row's further
  // entries, start << 4 | count, in the workgroup's xcol / xval
  const uint2 *lcol;
  const double *lval;
  const unsigned short *xcol;
  const double *xval;
  const int *x0;                         // first further entry of each workgroup (nblk + 1)
  const int *imp0, *exp0, *exp_row, *exp_slot;   // ghosts fetched, rows posted (null: uncoupled cells)
  unsigned long long wait;               // the limit of a wait (grid_mail.hpp)
  double *ghost;                         // [3][GHOST_STAGES][nslot]
  int nslot;
  double *terms, *parts;                 // grid_sum's mailboxes
  double *gap;                           // [3][n]: dendrite voltages for the olive's gap currents
  // Helpers: workgroups beyond nblk that only run ion updates, nhelp for each
  // of the others, which keeps the rows before own and gives every helper the
  // next own ones.  req [3][nblk][3]: the update's interval (< 0: the launch
  // ends), the macro step's time and the synaptic decay; vin, bout [3][nc]: the rows' new voltages
  // and their frozen currents.
  int nhelp, own;
  double *req, *vin, *bout;
  unsigned gq0;                          // number of the launch's first ion update
  double *y, *yn, *fn, *ede, *vnew, *b, *v1, *v2;
  const double *cm, *coef;               // coef: the coefficients, then {w1, mu~_1} of m = 0 .. RES_START stages
  // the record, and its copy in mapped host memory with a word behind it that
  // whichever workgroup or helper gives up sets
  RkcCtl *ctl, *ctl_host;
  // what stopped goes on: ASK_POW with err's powers p1, p2, ASK_STAGE with w1 and
  // mu~_1 in them, ASK_DECAY with the decay in p1 (0: nothing stopped)
  int resume;
  double p1, p2;
  double integ, rho_floor;
  int strict, refresh_fn;
  // per macro step: the stimulus, the Poisson drive, the recorder
  double *iext;
  const double *amp;
  int stim_comp, do_stim;
  double stim_t0, stim_t1;
  double *syn_g;                         // null: no drive
  double syn_decay, syn_p, syn_event;
  uint32_t k0, k1;
  double *rec;                           // this launch's recording, or null
  int rec_comp;                          // < 0: every compartment
  uint32_t *bits;
  double *prev;
  int raster_comp, words;
  double thr;
};

// x^(1/3) and x^(2/3) with the exponents 1.0 / 3.0 and 2.0 / 3.0 as the
// controller writes them: the cube root in double, its remainder by fused
// multiply-adds, and the factor x^(-d) for the exponent's own rounding
// d = 1/3 - fl(1/3) to first order; the error before the last rounding is
// below 1e-5 ulp.  The reference's controller rounds as the host's libm does,
// and at the granule cell's tolerance one last bit of a step size moves its
// voltage by 1e-4 mV within 0.5 ms.  libm's pow misses the nearest double only
// where the value lies within 0.0083 ulp of the middle between two (measured,
// 12 million arguments, 8e-4 of them missed), so a result that is POW_SLACK or more away from
// a middle is libm's result too; for the others (sure = false, one power in 50) the
// kernel stops and the host answers with pow: one attempt in 26 (olive) to 32 (granule,
// Golgi), since an accepted one needs both powers.
constexpr double POW_SLACK = 0.01;
struct CubeRoots {
  double p1, p2;
  bool sure1, sure2;
};
__device__ inline CubeRoots cube_roots(double x) {
  CubeRoots r;
  if (!(x > 1e-30 && x < 1e30)) {
    r.p1 = r.p2 = 0.0;
    r.sure1 = r.sure2 = false;
    return r;
  }
  const float l2 = __builtin_amdgcn_logf((float)x);
  double y = (double)__builtin_amdgcn_exp2f(l2 * (1.0f / 3.0f));   // relative error ~1e-6
  y = y - (y * y * y - x) / (3.0 * (y * y));                       // ~1e-12
  y = y - (y * y * y - x) / (3.0 * (y * y));                       // rounding level
  const double p = y * y, pe = fma(y, y, -p);
  const double q = p * y, qe = fma(p, y, -q);
  const double c = ((x - q) - qe - pe * y) / (3.0 * p);
  const double d = 1.850371707708594e-17 * ((double)l2 * 0.6931471805599453);
  r.p1 = round_sure(y, c - y * d, POW_SLACK, r.sure1);
  r.p2 = round_sure(p, pe + 2.0 * y * c - p * (2.0 * d), POW_SLACK, r.sure2);
  return r;
}

// The voltages behind the olive's explicit gap currents: a cell's dendrite in
// the workgroup's vector or in the mailbox
struct GapView {
  const double *y, *gap;
  int cell0, cells, comp;
  Wait *wait;
  __device__ double operator()(int cell) const {
    if (cell >= cell0 && cell < cell0 + cells) return y[(cell - cell0) * comp];
    return mail_get(gap + cell, *wait);
  }
};

// Model: NT threads, the state struct, ion(S, i, vn, dt, gap) = ion update and
// frozen current of row i (DECAY: with the synaptic current's decay over dt, which
// follows the host's libm like the powers of err: decay(dt) is its value, or NaN where
// it has to be asked), GAP = the olive's explicit gap currents, HELP = helpers
// may run it.  The
// update takes up to 430 registers, so nothing lives across it: the controller
// stays in LDS (a copy for every wave), the thread's matrix rows are read again
// after it, and it is inlined at one place only.

template <class Model>
__device__ __forceinline__ double model_ion(const typename Model::State *S, int i, double vn, double dt,
                                            const GapView *gap, double decay) {
  if constexpr (Model::DECAY) return Model::ion(S, i, vn, dt, gap, decay);
  else return Model::ion(S, i, vn, dt, gap);
}

// The ion updates of some of workgroup w's rows.  A cell of 1600 compartments
// is four rows to a thread of its workgroup, one after the other, while most
// CUs have nothing to do: 9 cells, 8 macro steps, 5.4 -> 3.9 ms with three
// helpers to a cell (16 granule cells with two, one step, 8.3 -> 7.0).  The
// mailbox protocol is grid_mail.hpp's with update numbers: what either side
// posted for update g - 1 is emptied after update g, and settled before it
// posts for g + 1.
template <class Model>
__device__ inline void rkc_helper(const RkcArgs &A, const typename Model::State *S, int w, int j, double *sm) {
  constexpr int NT = Model::NT;
  const int tid = threadIdx.x, RM = A.cpb * A.comp, R = min(RM, A.nc - w * RM);
  const int l0 = min(R, (j + 1) * A.own), l1 = min(R, l0 + A.own), r0 = w * RM;
  __shared__ int s_late;
  if (tid == 0) s_late = 0;
  Wait W{A.wait, &s_late, 0};
  for (unsigned g = A.gq0;; g = g == 2 ? 0 : g + 1) {
    if (tid == 0) {
      const double *rq = A.req + ((size_t)g * A.nblk + w) * 3;
      sm[0] = mail_wait(rq, W);
      sm[1] = mail_get(rq + 1, W);
      sm[2] = mail_get(rq + 2, W);
    }
    __syncthreads();
    const bool late = s_late;
    const double dt = sm[0], t = sm[1], decay = sm[2];
    __syncthreads();
    const size_t copy = (size_t)g * A.nc, old = (size_t)(g == 0 ? 2 : g - 1) * A.nc;
    mail_settle();
#pragma unroll 1
    for (int i = l0 + tid; i < l1; i += NT) {
      const int row = r0 + i;
      if (A.do_stim && row % A.comp == A.stim_comp)
        A.iext[row] = (A.stim_t0 <= t && t < A.stim_t1) ? A.amp[row / A.comp] : 0.0;
      if (!late && dt >= 0.0) {
        const double vn = mail_get(A.vin + copy + row, W);
        // without its voltages the helper posts nothing, and its workgroup gives up in turn
        if (!*W.late) mail_put(A.bout + copy + row, model_ion<Model>(S, row, vn, dt, nullptr, decay));
      }
      mail_clear(A.bout + old + row);
    }
    if (late || !(dt >= 0.0)) {
      if (late && tid == 0) *(int *)(A.ctl_host + 1) = 1;
      return;
    }
  }
}

// K: rows per thread (thread t owns rows t, t + NT, ...).  A thread's matrix
// rows, capacitances and frozen currents stay in its registers, so a stage
// reads the vectors only, all K rows' reads before the first use: from LDS,
// one row after the other, a stage of 1600 rows took 1.9 us.
template <class Model, int K>
__global__ void __launch_bounds__(Model::NT) k_rkc_steps(RkcArgs A, const typename Model::State *S, int nsteps, double t0,
                                                         int step0) {
  constexpr int NT = Model::NT;
  constexpr double UR = 2.22e-16, H = 0.125;
  extern __shared__ double sm[];
  const int tid = threadIdx.x, w = blockIdx.x;
  if constexpr (Model::HELP)
    if (w >= A.nblk) {
      rkc_helper<Model>(A, S, (w - A.nblk) / A.nhelp, (w - A.nblk) % A.nhelp, sm);
      return;
    }
  const bool helped = Model::HELP && A.nhelp > 0;
  const int cell0 = w * A.cpb, cells = min(A.cpb, A.n - cell0);
  const int r0 = cell0 * A.comp, R = cells * A.comp, RM = A.cpb * A.comp, RS = RM + A.ghost_max;
  double *Yv = sm, *YN = Yv + RS, *FN = YN + RS, *V1 = FN + RS, *V2 = V1 + RS;
  double *T = V2 + RS, *part = T + RM + RED_BLOCK, *C4 = part + A.nch + 8, *XV = C4 + 4 * RES_COEF;
  unsigned short *XC = (unsigned short *)(XV + A.ext_max);
  __shared__ int s_late;
  if (tid == 0) s_late = 0;
  Wait W{A.wait, &s_late, 0};
  bool late = false;   // the same in the whole workgroup: a wait gave up before the last sum or ion update
  SumPlan P;
  P.set(A.nc, r0, r0 + R);

  RkcCtl *ctl = A.ctl;
  const double at = ctl->o[4], rt = ctl->o[5], hmin = ctl->hw[6], mmax = ctl->o[0];
  __shared__ double s_ctl[NT / 64][16];
  __shared__ int s_m;              // stages of the attempt that the host is asked about: thread 0's
  __shared__ long long s_cnt[5];   // steps, rejects, stages, power iterations, ion updates: kept by thread 0
  double *cs = s_ctl[tid >> 6];
  double &absh = cs[0], &sprad = cs[1], &naccpt = cs[2], &idid = cs[3], &gt = cs[4], &gt_old = cs[5], &lt = cs[6],
         &tend = cs[7], &errold = cs[8], &hold = cs[9], &hw0 = cs[10], &hw1 = cs[11], &sum_dt = cs[12], &err = cs[13],
         &errold3 = cs[14], &h_now = cs[15];
  absh = ctl->o[1]; sprad = ctl->o[2]; naccpt = ctl->o[3]; idid = ctl->o[6]; gt = ctl->o[7]; gt_old = ctl->o[8];
  lt = ctl->o[9]; tend = ctl->o[10]; errold = ctl->o[11]; hold = ctl->o[12]; hw0 = ctl->hw[0]; hw1 = ctl->hw[1];
  sum_dt = ctl->sum_dt; err = ctl->err; errold3 = ctl->errold3; h_now = ctl->h;
  if (tid == 0) {
    s_cnt[0] = ctl->steps; s_cnt[1] = ctl->rejects; s_cnt[2] = ctl->stages; s_cnt[3] = ctl->rho_iters;
    s_cnt[4] = ctl->ions;
  }
  auto count = [&](int k, int n) {
    if (tid == 0) s_cnt[k] += n;
  };
  bool last = ctl->last, newspc = ctl->newspc, jacatt = ctl->jacatt;
  unsigned q = ctl->q, gq = A.gq0;
  int status = 0, done_steps = 0;
  int resume = A.resume;
  int loops = ctl->loops;
  CubeRoots ce;
  ce.p1 = A.p1;
  ce.p2 = A.p2;

  // the workgroup's rows
  double cm[K], bb[K], wt3[K][ROW_W];
  uint2 nb[K];
  {
    const int x0 = A.x0[w], nx = A.x0[w + 1] - x0;
    for (int k = tid; k < nx; k += NT) {
      XV[k] = A.xval[x0 + k];
      XC[k] = A.xcol[x0 + k];
    }
    for (int i = tid; i < R; i += NT) {
      Yv[i] = A.y[r0 + i];
      YN[i] = A.yn[r0 + i];
      FN[i] = A.fn[r0 + i];
      T[i] = A.b[r0 + i];
      if (resume == ASK_POW) {
        V1[i] = A.v1[r0 + i];
        V2[i] = A.v2[r0 + i];
      }
    }
  }
  // the thread's matrix rows and capacitances, and its frozen currents from T
  auto load_rows = [&]() {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int i = tid + k * NT;
      cm[k] = 1.0;
      bb[k] = 0.0;
      nb[k] = make_uint2(0u, 0u);
#pragma unroll
      for (int e = 0; e < ROW_W; e++) wt3[k][e] = 0.0;
      if (i < R) {
        bb[k] = T[i];
        cm[k] = A.cm[r0 + i];
        nb[k] = A.lcol[r0 + i];
#pragma unroll
        for (int e = 0; e < ROW_W; e++) wt3[k][e] = A.lval[(size_t)e * A.nc + r0 + i];
      }
    }
  };
  load_rows();
  __syncthreads();

  // F(y) of the thread's k-th row, its sum in column order; a missing
  // neighbour is the row itself with conductance 0 (adds an exact zero)
  auto rhs = [&](int k, double yi, const double *y) {
    double d = -bb[k];
    d += wt3[k][0] * (y[nb[k].x & 0xFFFFu] - yi);
    d += wt3[k][1] * (y[nb[k].x >> 16] - yi);
    d += wt3[k][2] * (y[nb[k].y & 0xFFFFu] - yi);
    const unsigned x = nb[k].y >> 16;
    if (x & 15u)
      for (unsigned j = x >> 4, e = j + (x & 15u); j < e; j++) d += XV[j] * (y[XC[j]] - yi);
    return d / cm[k];
  };
  // f(k, i) for the thread's rows
  auto rows = [&](auto f) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int i = tid + k * NT;
      if (i < R) f(k, i);
    }
  };
  auto total = [&]() { return grid_sum<NT>(P, T, part, A.terms, A.parts, q, W, late); };
  // coupled cells: the neighbours' compartments of vector v into its tail.
  // Every exchange between two sums has slots of its own; they are emptied
  // like the sum's, after the next one.
  int gs = ctl->ghost_now, gs_old = ctl->ghost_used;
  const bool coupled = A.imp0 != nullptr;
  auto finish_sum = [&]() {
    const double s = total();
    if (coupled) {
      double *old = A.ghost + (size_t)(q == 2 ? 0 : q + 1) * GHOST_STAGES * A.nslot;   // of the sum before this one
      const int e0 = A.exp0[w], ne = A.exp0[w + 1] - e0;
      for (int k = tid; k < ne * gs_old; k += NT) mail_clear(old + (size_t)(k / ne) * A.nslot + A.exp_slot[e0 + k % ne]);
      gs_old = gs;
      gs = 0;
    }
    return s;
  };
  auto fetch = [&](double *v) {
    if (!coupled) return;
    double *g = A.ghost + ((size_t)q * GHOST_STAGES + gs) * A.nslot;
    for (int k = A.exp0[w] + tid; k < A.exp0[w + 1]; k += NT) mail_put(g + A.exp_slot[k], v[A.exp_row[k]]);
    const int m0 = A.imp0[w], ni = A.imp0[w + 1] - m0;
    for (int k = tid; k < ni; k += NT) v[R + k] = mail_get(g + m0 + k, W);
    gs++;
    __syncthreads();
  };

  // an ion update for the helpers, and the emptying of the one before it
  double t_now = t0;
  auto request = [&](double dt, int own, double decay) {
    mail_settle();
    __syncthreads();
    for (int i = own + tid; i < R && dt >= 0.0; i += NT) mail_put(A.vin + (size_t)gq * A.nc + r0 + i, Yv[i]);
    if (tid < 3) mail_put(A.req + ((size_t)gq * A.nblk + w) * 3 + tid, tid == 0 ? dt : tid == 1 ? t_now : decay);
  };
  auto forget = [&](int own) {
    const size_t old = gq == 0 ? 2 : gq - 1;
    for (int i = own + tid; i < R; i += NT) mail_clear(A.vin + old * A.nc + r0 + i);
    if (tid < 3) mail_clear(A.req + (old * A.nblk + w) * 3 + tid);
  };
  auto ion_and_b = [&](double dt, double decay) {
    count(4, 1);
    if constexpr (Model::GAP) {
      // the dendrites' new voltages, for the gap currents of other workgroups' cells
      if (!P.alone) {
        for (int c = tid; c < cells; c += NT) {
          mail_clear(A.gap + (size_t)(gq == 2 ? 0 : gq + 1) * A.n + cell0 + c);
          mail_put(A.gap + (size_t)gq * A.n + cell0 + c, Yv[c * A.comp]);
        }
      }
    }
    const GapView gv{Yv, A.gap + (size_t)gq * A.n, cell0, cells, A.comp, &W};
    const int own = helped ? min(R, A.own) : R;
    if (helped) request(dt, own, decay);
#pragma unroll 1
    for (int i = tid; i < own; i += NT) T[i] = model_ion<Model>(S, r0 + i, Yv[i], dt, &gv, decay);
    if (helped) {
      for (int i = own + tid; i < R; i += NT) T[i] = mail_get(A.bout + (size_t)gq * A.nc + r0 + i, W);
      forget(own);
      __syncthreads();   // T's rows change threads here
    }
    load_rows();
    gq = gq == 2 ? 0 : gq + 1;
    if (A.refresh_fn) {
      __syncthreads();
      fetch(YN);
      rows([&](int k, int i) { FN[i] = rhs(k, YN[i], YN); });
    }
    late = __syncthreads_or(W.mine);
  };

  // rkcrho (solve_rkc.cu:562-754)
  auto rkcrho = [&]() {
    const int itmax = 1000;
    double so[3] = {0.0, 0.0, 0.0};
    const double sqrtu = sqrt(UR), small = 1.0 / 0.125;
    double ynrm = 0.0, vnrm = 0.0, dynrm;
#pragma unroll 1
    for (int n = 0; n < 2; n++) {
      for (int i = tid; i < R; i += NT) {
        const double v = n == 0 ? YN[i] : A.ede[r0 + i];
        T[i] = v * v;
      }
      ynrm = vnrm;
      vnrm = sqrt(finish_sum());
    }
    if (ynrm != 0.0 && vnrm != 0.0) {
      dynrm = ynrm * sqrtu;
      const double f = dynrm / vnrm;
      for (int i = tid; i < R; i += NT) V1[i] = f * A.ede[r0 + i] + YN[i];
    } else if (ynrm != 0.0) {
      dynrm = ynrm * sqrtu;
      for (int i = tid; i < R; i += NT) V1[i] = sqrtu * YN[i] + YN[i];
    } else if (vnrm != 0.0) {
      dynrm = UR;
      const double f = dynrm / vnrm;
      for (int i = tid; i < R; i += NT) V1[i] = f * A.ede[r0 + i];
    } else {
      dynrm = UR;
      for (int i = tid; i < R; i += NT) V1[i] = dynrm;
    }
    double sigma = 0.0, sigmal;
    for (int iter = 0; iter < itmax && !late; iter++) {
      count(3, 1);
      __syncthreads();
      fetch(V1);
      rows([&](int k, int i) {
        const double F = rhs(k, V1[i], V1);
        V2[i] = F;
        const double d = -1.0 * FN[i] + F;
        T[i] = d * d;
      });
      const double dfnrm = sqrt(finish_sum());
      sigmal = sigma;
      sigma = dfnrm / dynrm;
      so[0] = so[1];
      so[1] = so[2];
      so[2] = sprad;
      sprad = 1.2 * sigma;
      bool done = iter >= 1 && fabs(sigma - sigmal) <= ((sigma > small) ? sigma : small) * 0.001;
      if (!done && iter > itmax / 2 && fabs(so[2] - so[0]) < 0.00001 && fabs(so[1] - sprad) < 0.00001) {
        sprad = (sprad + so[2]) / 2.0;
        done = true;
      }
      if (done) {
        for (int i = tid; i < R; i += NT) A.ede[r0 + i] = -1.0 * YN[i] + V1[i];
        return;
      }
      if (dfnrm != 0.0) {
        const double al = dynrm / dfnrm;
        for (int i = tid; i < R; i += NT) {
          const double t = -1.0 * V2[i] + FN[i];
          V1[i] = al * t + YN[i];
        }
      } else {
        const int id = iter % A.nc - r0;
        if (id >= 0 && id < R && id % NT == tid) V1[id] = 2.0 * YN[id] - V1[id];
      }
    }
    idid = 6;
  };

  // step (solve_rkc.cu:815-906)
  auto step = [&](double h, int m) {
    double w0 = 0.0, w1 = 0.0, mus;
    const bool tab = m >= 2 && m <= RES_COEF;
    if (tab) {
      const double *ct = A.coef + (size_t)m * RES_COEF * 4;
      for (int k = tid; k < 4 * m; k += NT) C4[k] = ct[k];
      mus = ct[0];
    } else {
      w0 = 1.0 + 2.0 / (13.0 * m * m);
      w1 = m > RES_START ? A.p1 : A.coef[RES_COEFS + 2 * m];
      mus = m > RES_START ? A.p2 : A.coef[RES_COEFS + 2 * m + 1];
    }
    const double hm = h * mus;
    for (int i = tid; i < R; i += NT) {
      const double y0 = YN[i];
      V2[i] = y0;
      V1[i] = hm * FN[i] + y0;
    }
    count(2, m);
    __syncthreads();
    double bjm1 = 1.0 / ((2.0 * w0) * (2.0 * w0)), bjm2 = bjm1;
    double zjm1 = w0, zjm2 = 1.0, dzjm1 = 1.0, dzjm2 = 0.0, d2zjm1 = 0.0, d2zjm2 = 0.0;
    for (int j = 1; j < m; j++) {
      double mu, nu, ajm1;
      if (tab) {
        mu = C4[4 * j];
        nu = C4[4 * j + 1];
        mus = C4[4 * j + 2];
        ajm1 = C4[4 * j + 3];
      } else {
        const double zj = 2.0 * w0 * zjm1 - zjm2, dzj = 2.0 * w0 * dzjm1 - dzjm2 + 2.0 * zjm1;
        const double d2zj = 2.0 * w0 * d2zjm1 - d2zjm2 + 4.0 * dzjm1;
        const double bj = d2zj / (dzj * dzj);
        ajm1 = 1.0 - zjm1 * bjm1;
        mu = 2.0 * w0 * bj / bjm1;
        nu = -bj / bjm2;
        mus = mu * w1 / w0;
        bjm2 = bjm1; bjm1 = bj;
        zjm2 = zjm1; zjm1 = zj;
        dzjm2 = dzjm1; dzjm1 = dzj;
        d2zjm2 = d2zjm1; d2zjm1 = d2zj;
      }
      const double omn = 1.0 - mu - nu, hs = h * mus;
      if (coupled && gs >= GHOST_STAGES - 2) {   // nearly out of slots: a sum of nothing in between
        for (int i = tid; i < R; i += NT) T[i] = 0.0;
        finish_sum();
      }
      fetch(V1);
      // every row's reads before the first division: without a value kept
      // apart the compiler orders a row's store before the next row's reads
      double yo[K];
      rows([&](int k, int i) {
        const double v1 = V1[i];
        const double F = rhs(k, v1, V1);
        yo[k] = mu * v1 + nu * V2[i] + omn * YN[i] + hs * (F - ajm1 * FN[i]);
      });
      rows([&](int k, int i) { Yv[i] = yo[k]; });
      double *t = V2;
      V2 = V1;
      V1 = Yv;
      Yv = t;
      __syncthreads();
    }
    double *t = Yv;
    Yv = V1;
    V1 = V2;
    V2 = t;
  };

  // an attempt of rkclow (solve_rkc.cu:908-1096) up to its error norm
  auto attempt = [&]() {
    if (newspc) {
      rkcrho();
      if (late) return;   // (the estimate is of no use, and could ask for thousands of stages)
      if (sprad < A.rho_floor) sprad = A.rho_floor;
      jacatt = true;
    }
    const double absh_in = absh;
    last = false;
    if (1.1 * absh >= fabs(tend - lt)) {
      absh = fabs(tend - lt);
      last = true;
    }
    const double mr = sqrt(1.54 * absh * sprad + 1.0);
    int m = (mr < mmax) ? 1 + (int)mr : (int)mmax + 1;
    if (m > mmax) {
      m = (int)mmax;
      absh = (m * m - 1) / (1.54 * sprad);
      last = false;
    }
    if (__builtin_expect(m > RES_START && !resume, 0)) {   // the attempt begins again, but for the spectral radius
      absh = absh_in;
      newspc = false;
      status = ASK_STAGE;
      if (tid == 0) s_m = m;
      return;
    }
    double h = absh;
    if (h <= hmin) h = hmin;
    h_now = h;
    step(h, m);
    // f(Y_m) and the error estimate (every weight is positive: atol > 0)
    fetch(Yv);
    double fo[K], to[K];
    rows([&](int k, int i) {
      const double yi = Yv[i], yni = YN[i];
      const double F = rhs(k, yi, Yv);
      const double ay = fabs(yi), ayn = fabs(yni);
      const double wt = at + rt * ((ay > ayn) ? ay : ayn);
      const double est = 0.8 * (yni - yi) + 0.4 * h * (FN[i] + F);
      fo[k] = F;
      to[k] = (est / wt) * (est / wt);
    });
    rows([&](int k, int i) {
      V1[i] = fo[k];
      T[i] = to[k];
    });
    count(2, 1);
    err = sqrt(finish_sum() / (double)A.nc);
  };

  auto rkclow = [&]() {
    if (!resume) loops = 0;
    while (!late) {
      if (resume == ASK_POW) {
        resume = 0;
      } else {
        if (!resume && ++loops > 1000) return;
        attempt();
        resume = 0;
        if (late || status != 0) return;
        if (!isfinite(err)) {
          status = Model::NONFINITE_STATUS;
          return;
        }
        ce = cube_roots(err);
        // err^(2/3) enters an accepted step's factor only
        const bool accepts = err <= 1.0 || !ce.sure1 || 0.8 * absh / ce.p1 < hmin;
        if (!ce.sure1 || (accepts && !ce.sure2)) {
          status = ASK_POW;
          return;
        }
      }
      const double h = h_now;
      if (err > 1.0) {
        count(1, 1);
        absh = 0.8 * absh / ce.p1;
        if (absh < hmin) {
          idid = 4;   // and fall through to the accept branch, as the reference does
        } else {
          newspc = !jacatt;
          continue;
        }
      }
      count(0, 1);
      naccpt += 1;
      lt += h;
      gt = lt;
      jacatt = false;
      newspc = false;   // nstsig is never advanced in the reference
      hw0 = h;
      hw1 = lt;
      double *t = V2;
      V2 = FN;
      FN = V1;
      V1 = YN;
      YN = Yv;
      Yv = t;
      double fac = 10.0, t1, t2;
      if (naccpt == 1) {
        t2 = ce.p1;
        if (0.8 < fac * t2) fac = 0.8 / t2;
      } else {
        t1 = 0.8 * absh * errold3;
        t2 = fabs(hold) * ce.p2;
        if (t1 < fac * t2) fac = t1 / t2;
      }
      absh = ((0.1 > fac) ? 0.1 : fac) * absh;
      const double hm = fmin(H, absh);
      absh = (hmin > hm) ? hmin : hm;
      errold = err;
      errold3 = ce.p1;
      hold = h;
      idid = last ? 1 : 2;
      return;
    }
  };

  for (int s = 0; s < nsteps; s++) {
    const double t = t0 + s * H;
    t_now = t;
    for (int i = tid; i < R && !resume; i += NT) {
      const int cell = (r0 + i) / A.comp, k = r0 + i - cell * A.comp;
      if (A.do_stim && k == A.stim_comp && (!helped || i < A.own)) A.iext[r0 + i] = (A.stim_t0 <= t && t < A.stim_t1) ? A.amp[cell] : 0.0;
      if (A.syn_g) {
        const u32x4 r = philox4x32_10((uint32_t)(r0 + i), (uint32_t)(step0 + s), 0x5359u, 0u, A.k0, A.k1);
        const double u = u01_53(r.v[0], r.v[1]);
        A.syn_g[r0 + i] = A.syn_g[r0 + i] * A.syn_decay + ((u < A.syn_p) ? A.syn_event : 0.0);
      }
    }
    bool ion_due = sum_dt != 0.0 && (!resume || resume == ASK_DECAY);
    while (true) {
      if (ion_due) {
        double decay = 0.0;
        if constexpr (Model::DECAY)
          if (S->net_s) {
            decay = resume ? A.p1 : Model::decay(sum_dt);
            resume = 0;
            if (!(decay == decay)) {
              status = ASK_DECAY;
              break;
            }
          }
        ion_and_b(sum_dt, decay);
        sum_dt = 0.0;
        ion_due = false;
      }
      rkclow();
      if (late || status != 0) break;
      sum_dt += gt - gt_old;
      gt_old = gt;
      ion_due = (A.strict ? sum_dt > A.integ : sum_dt >= A.integ) && idid == 2.0;
      if (idid == 2.0) continue;
      if (idid == 1.0) break;
      status = (int)idid;
      break;
    }
    if (late) status = TIMED_OUT;
    if (status != 0) break;
    // rkcint at gt_old (solve_rkc.cu:794-813), the recorder and the raster
    const double tlast = hw1 - hw0, x = (gt_old - tlast) / hw0;
    const double a1 = (1.0 + 2.0 * x) * (x - 1.0) * (x - 1.0), a2 = (3.0 - 2.0 * x) * x * x;
    const double b1 = hw0 * x * (x - 1.0) * (x - 1.0), b2 = hw0 * (x - 1.0) * x * x;
    for (int i = tid; i < R; i += NT) {
      const double v = a1 * V1[i] + a2 * YN[i] + b1 * V2[i] + b2 * FN[i];
      const int cell = (r0 + i) / A.comp, k = r0 + i - cell * A.comp;
      A.vnew[r0 + i] = v;
      if (A.rec) {
        if (A.rec_comp < 0) A.rec[(size_t)s * A.nc + r0 + i] = v;
        else if (k == A.rec_comp) A.rec[(size_t)s * A.n + cell] = v;
      }
      if (A.bits && k == A.raster_comp) {
        if (v > A.thr && A.prev[cell] <= A.thr) atomicOr(&A.bits[(size_t)s * A.words + (cell >> 5)], 1u << (cell & 31));
        A.prev[cell] = v;
      }
    }
    tend += H;
    done_steps++;
  }

  if (helped) {
    request(-1.0, R, 0.0);
    forget(min(R, A.own));
    gq = gq == 2 ? 0 : gq + 1;
  }
  rows([&](int k, int i) {
    A.y[r0 + i] = Yv[i];
    A.yn[r0 + i] = YN[i];
    A.fn[r0 + i] = FN[i];
    A.b[r0 + i] = bb[k];
    if (status == ASK_POW) {
      A.v1[r0 + i] = V1[i];
      A.v2[r0 + i] = V2[i];
    }
  });
  if (tid == 0 && s_late) *(int *)(A.ctl_host + 1) = 1;
  if (w == 0 && tid == 0) {
    RkcCtl c = *ctl;
    c.o[1] = absh; c.o[2] = sprad; c.o[3] = naccpt; c.o[6] = idid; c.o[7] = gt;
    c.o[8] = gt_old; c.o[9] = lt; c.o[10] = tend; c.o[11] = errold; c.o[12] = hold;
    c.hw[0] = hw0; c.hw[1] = hw1;
    c.sum_dt = sum_dt; c.errold3 = errold3; c.err = err; c.h = h_now;
    c.steps = s_cnt[0]; c.rejects = s_cnt[1]; c.stages = s_cnt[2]; c.rho_iters = s_cnt[3]; c.ions = s_cnt[4];
    c.macro += done_steps;
    c.last = last; c.newspc = newspc; c.jacatt = jacatt; c.status = status;
    c.q = q; c.ions_q = gq; c.ghost_used = gs_old; c.loops = loops; c.m = s_m; c.ghost_now = gs;
    *ctl = c;
    *A.ctl_host = c;
  }
}

}  // namespace cbrkc

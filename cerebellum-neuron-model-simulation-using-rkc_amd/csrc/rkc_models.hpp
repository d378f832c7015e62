// The cell types on the population-global RKC path: each one's ion update with
// its frozen current (used by the launch-per-stage kernels too), and its model
// for the resident kernel.  The kernels of a model are compiled by a file of
// their own (rkc_pkj.hip, ...), side by side: together they took four minutes.
#pragma once
#include <hip/hip_runtime.h>

#include "engine.hpp"
#include "ion_state.hpp"
#include "pkj_model.hpp"
#include "rkc_resident.hpp"

namespace cbrkc {

struct PkjState {
  double *v, *ca, *rev, *iext, *shell;
  const double *cond;   // [NCOND][nc]
  double *gate;         // [NGATE][nc]
  double *b;
  const double *syn_g;  // may be null
  double syn_e;
  int nc;
  const double *net_s;  // synaptic current of the macro step (granule input), may be null
  double net_decay;     // exp(-dt / 0.6), dt the ion interval, as the host's libm gives it
};

// pkj_update_ion_RKC (pkj_ion.cu:304-358) followed by pkj_update_matrix
// (solve_rkc.cu:369-395), fused: one pass over the compartment state.
// With do_ion == 0 only the current is rebuilt (RKC_vec_initialize).
__device__ inline double pkj_ion_current(const PkjState &S, int i, double vn, double DT, bool do_ion) {
  using namespace pkj;
  const int nc = S.nc;
  double g[NGATE], c[NCOND];
#pragma unroll
  for (int k = 0; k < NGATE; k++) g[k] = S.gate[(size_t)k * nc + i];
#pragma unroll
  for (int k = 0; k < NCOND; k++) c[k] = S.cond[(size_t)k * nc + i];
  double rev = S.rev[i];
  if (do_ion) {
    const double vo = S.v[i];
    const double vm = 0.5 * (vn + vo);
    double ca = S.ca[i];
    double caq = ca_rk4(vo, ca, rev, S.shell[i], c[g_CaP] * g[m_CaP] * g[h_CaP], c[g_CaT] * g[m_CaT] * g[h_CaT], DT,
                        i % 1599 == 0);
    gates_cn<double>(vm, caq, DT, g);
#pragma unroll
    for (int k = 0; k < NGATE; k++) S.gate[(size_t)k * nc + i] = g[k];
    S.ca[i] = ca;
    S.rev[i] = rev;
    S.v[i] = vn;
  }
  double bb = current<double>(vn, S.iext[i], rev, c, g);
  if (S.syn_g) bb += S.syn_g[i] * (vn - S.syn_e);
  // pkj_update_matrix_new (solve_rkc.cu:358-367, 1245-1249)
  if (S.net_s) bb += S.net_s[i] * S.net_decay;
  return bb;
}

// io_update_ion_RKC (io_ion.cu:90-127), io_update_matrix (solve_rkc.cu:412-434)
// and, on each dendrite, the gap currents of io_gap_update / add_io_gap_val
// (gap.cu:149-160, solve_rkc.cu:400-410), fused.  The gap current uses the
// partners' voltages after the update (elem[v] = vnew there) and is added in
// partner order 0..3 (the reference adds with atomics in no fixed order).
// dend(cell): the new voltage of a cell's dendrite.
template <class Dend>
__device__ inline double io_ion_gap_current(const IoState &S, int i, double vn, double DT, bool do_ion, Dend dend) {
  using namespace io;
  double bb = io_ion_current(S, i, vn, DT, do_ion);
  if (do_ion && S.n > 1 && i % COMP == 0) {
    const int cell = i / COMP;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int pre = S.nbr[cell * 4 + s];
      const double diff_v = (pre > -1) ? (vn - dend(pre)) : 0.0;
      bb += gap_current<double>(diff_v);
    }
  }
  if (S.syn_g) bb += S.syn_g[i] * (vn - S.syn_e);
  return bb;
}

// go_update_ion_RKC_exp_imp (go_ion.cu:379-437), go_KAHP_update_2order
// (go_ion.cu:88-213) and go_update_matrix (solve_rkc.cu:288-314), fused: the
// three reference kernels touch one compartment's state each, in this order
// (solve_rkc.cu:1174-1179).  The intercell gap junctions are in the cable
// matrix, not here.
__device__ inline double go_ion_net_current(const GoState &S, int i, double vn, double DT, bool do_ion) {
  double bb = go_ion_current(S, i, vn, DT, do_ion);
  if (S.syn_g) bb += S.syn_g[i] * (vn - S.syn_e);
  // go_update_matrix_new (solve_rkc.cu:279-286, 1181)
  if (S.net_s) bb += S.net_s[i];
  return bb;
}

// gr_Na_update_2order (gr_ion.cu:45-207), gr_update_ion_RKC_exp_imp
// (gr_ion.cu:461-480) and gr_update_matrix (solve_rkc.cu:226-249), fused in
// the reference's order (solve_rkc.cu:1111-1116): the Na scheme sees the
// voltage of the previous ion update and the new one, then the gates move and
// the stored voltage becomes the new one.
__device__ inline double gr_ion_net_current(const GrState &S, int i, double vn, double DT, bool do_ion) {
  double bb = gr_ion_current(S, i, vn, DT, do_ion);
  if (S.syn_g) bb += S.syn_g[i] * (vn - S.syn_e);
  // add_mfgr_val / add_gogr_val (solve_rkc.cu:200-224, 1117-1118), one
  // synapse after the other
  if (S.net.on())
    for (int j = S.net.row[i]; j < S.net.row[i + 1]; j++) {
      double E;
      const double gs = syn_entry(S.net, j, E);
      bb += gs * (vn - E);
    }
  return bb;
}

// The models of the resident kernel.  512 threads hold a Purkinje cell's 1600
// compartments four to a thread; the granule and Golgi updates keep their 12 x 12
// and 6 x 6 systems in registers, which takes one wave per SIMD.  K0 <= K1 <= K2:
// the rows per thread a kernel is built for (0: none).
struct PkjModel {
  using State = PkjState;
  static constexpr int NT = 512, K0 = 0, K1 = 0, K2 = 4, NONFINITE_STATUS = NONFINITE;
  static constexpr bool GAP = false, HELP = true, DECAY = true;
  // (a call, so that populations without synapses do not pay for it in registers)
  __device__ __attribute__((noinline)) static double decay(double dt) {
    bool sure;
    const double d = exp_libm(-dt / 0.6, sure);
    return sure ? d : __longlong_as_double(0x7FF8000000000000ll);
  }
  __device__ __attribute__((noinline)) static double ion(const State *Sp, int i, double vn, double dt, const GapView *,
                                                         double decay) {
    State S = *Sp;
    S.net_decay = decay;
    return pkj_ion_current(S, i, vn, dt, true);
  }
};
struct IoModel {
  using State = IoState;
  static constexpr int NT = 256, K0 = 0, K1 = 1, K2 = 7, NONFINITE_STATUS = NONFINITE;
  static constexpr bool GAP = true, HELP = false, DECAY = false;
  __device__ __forceinline__ static double ion(const State *S, int i, double vn, double dt, const GapView *gap) {
    return io_ion_gap_current(*S, i, vn, dt, true, [&](int cell) { return (*gap)(cell); });
  }
};
struct GoModel {
  using State = GoState;
  static constexpr int NT = 256, K0 = 0, K1 = 1, K2 = 7, NONFINITE_STATUS = NONFINITE;
  static constexpr bool GAP = false, HELP = false, DECAY = false;
  __device__ __forceinline__ static double ion(const State *S, int i, double vn, double dt, const GapView *) {
    return go_ion_net_current(*S, i, vn, dt, true);
  }
};
struct GrModel {
  using State = GrState;
  static constexpr int NT = 256, K0 = 1, K1 = 3, K2 = 7, NONFINITE_STATUS = NONFINITE;
  static constexpr bool GAP = false, HELP = true, DECAY = false;
  __device__ __attribute__((noinline)) static double ion(const State *S, int i, double vn, double dt, const GapView *) {
    return gr_ion_net_current(*S, i, vn, dt, true);
  }
};

// the model's kernel for k rows per thread: the next of its shapes
template <class Model>
const void *rkc_kernel_of(int k) {
  if constexpr (Model::K0 > 0)
    if (k <= Model::K0) return (const void *)k_rkc_steps<Model, Model::K0>;
  if constexpr (Model::K1 > 0)
    if (k <= Model::K1) return (const void *)k_rkc_steps<Model, Model::K1>;
  return (const void *)k_rkc_steps<Model, Model::K2>;
}
const void *rkc_kernel_pkj(int k);
const void *rkc_kernel_io(int k);
const void *rkc_kernel_go(int k);
const void *rkc_kernel_gr(int k);

}  // namespace cbrkc

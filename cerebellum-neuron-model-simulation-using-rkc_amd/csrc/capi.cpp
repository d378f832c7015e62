// extern "C" boundary of libcbrkc.so (declared in include/cbrkc.h).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <string>

#include "../../include/cbrkc.h"
#include "engine.hpp"
#include "go_model.hpp"
#include "gr_model.hpp"
#include "io_model.hpp"
#include "morph.hpp"
#include "network.hpp"
#include "philox.hpp"
#include "pkj_model.hpp"

using namespace cbrkc;

struct cb_syn;

struct cb_pop {
  std::unique_ptr<Engine> eng;
  int cell_type = CB_PKJ;
  int solver = CB_SOLVER_RKC;
  int engine = CB_ENGINE_GLOBAL_FP64;
  int comp = 0;
  int device = 0;
  int nx = 0, ny = 0;
  // incoming synapse sets (at most two: granule cells take mossy-fibre and
  // Golgi input) and their CSR by postsynaptic compartment on the device
  std::vector<cb_syn *> syn_in;
  int *syn_row = nullptr, *syn_slot = nullptr;
  // coupled to a network (cb_net), which holds its engine
  bool in_net = false;
  ~cb_pop() {
    eng.reset();
    if (syn_row) (void)hipFree(syn_row);
    if (syn_slot) (void)hipFree(syn_slot);
  }
};

// one synapse set (the reference's synapse_t, syn.cuh:76-82) on the device
struct cb_syn {
  SynHost host;
  cb_pop *pre = nullptr, *post = nullptr;
  int *pre_d = nullptr;
  double *x_d[3] = {nullptr, nullptr, nullptr};
  double *w_d = nullptr, *val_d = nullptr, *old_d = nullptr;
  uint64_t seed = 0;
  uint32_t step = 0;
  int device = 0;
  ~cb_syn() {
    for (void *p : {(void *)pre_d, (void *)x_d[0], (void *)x_d[1], (void *)x_d[2], (void *)w_d, (void *)val_d,
                    (void *)old_d})
      if (p) (void)hipFree(p);
  }
};


namespace {
thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

template <typename F>
int guarded(F &&f) {
  try {
    g_err.clear();
    return f();
  } catch (const Error &e) {
    g_err = e.msg;
    if (e.msg.rfind("HIP error", 0) == 0) return CB_E_HIP;
    if (e.code > 0) return CB_E_SOLVER;
    if (e.code == CB_E_UNSUP || e.code == CB_E_HIP) return e.code;
    return CB_E_ARG;
  } catch (const std::exception &e) {
    g_err = e.what();
    return CB_E_ARG;
  }
}

PoissonSpec poisson_of(const cb_pop_config &cfg) {
  PoissonSpec syn;
  syn.on = cfg.poisson_on != 0;
  syn.rate_hz = cfg.poisson_rate_hz;
  syn.g_event = cfg.poisson_g_mS;
  syn.tau_ms = cfg.poisson_tau_ms;
  syn.e_syn = cfg.poisson_e_mV;
  syn.seed = cfg.poisson_seed;
  return syn;
}

// io_initialize + io_solve_initialize + io_gap_create (io.cu:186-229,
// io_solve.cu:192-262, gap.cu:136-147): global FP64 engine only
int create_io(const cb_pop_config &cfg, cb_pop **out) {
  const int n = cfg.nx * cfg.ny;
  if (n == 0) return fail(CB_E_ARG, "empty population");
  if (cfg.engine != CB_ENGINE_GLOBAL_FP64 && cfg.engine != CB_ENGINE_TREE_FP64)
    return fail(CB_E_UNSUP, "inferior-olive cells are gap-junction coupled: global engine only");
  IoHost host;
  std::string err;
  const std::string path = cfg.morph_path ? cfg.morph_path : "./IO.txt";
  if (!build_io_host(path, cfg.nx, cfg.ny, cfg.v0, host, err)) return fail(CB_E_IO, err);
  StimSpec stim;   // io_set_current (io.cu:247-257): the dendrite, [800, 820) ms
  stim.comp = 0;
  stim.t0 = io::STIM_T0;
  stim.t1 = io::STIM_T1;
  if (cfg.stim_comp >= 0) {
    if (cfg.stim_comp >= io::COMP) return fail(CB_E_ARG, "stimulus compartment out of range");
    stim.comp = cfg.stim_comp;
    stim.t0 = cfg.stim_t0;
    stim.t1 = cfg.stim_t1;
  }
  stim.amp.assign(n, io::STIM);
  if (cfg.stim_amp)
    for (int c = 0; c < n; c++) stim.amp[c] = cfg.stim_amp[c];
  if (cfg.stim_comp == CB_STIM_NONE) stim.amp.assign(n, 0.0);
  SolverSpec sol;
  const double tol = 1.0e-6;   // TOL_IO, solve_rkc.cuh:31
  sol.atol = cfg.atol > 0 ? cfg.atol : tol;
  sol.rtol = cfg.rtol > 0 ? cfg.rtol : tol;
  sol.ion_interval = cfg.ion_interval_ms;
  sol.hmin = cfg.hmin_ms;
  sol.refresh_fn = cfg.refresh_fn != 0;
  if (cfg.rho_floor) return fail(CB_E_UNSUP, "the spectral-radius floor is provided for Purkinje cells");
  if (!(sol.atol > 0.0) || !(sol.rtol >= 0.0)) return fail(CB_E_ARG, "atol must be > 0 and rtol >= 0");
  std::unique_ptr<cb_pop> p(new cb_pop);
  p->cell_type = CB_IO;
  p->solver = cfg.solver;
  p->engine = cfg.engine;
  p->comp = io::COMP;
  p->device = cfg.device;
  CB_HIP(hipSetDevice(cfg.device));
  const bool tree = cfg.engine == CB_ENGINE_TREE_FP64;
  if (cfg.solver == CB_SOLVER_CN)
    p->eng.reset(make_cn_io(host, stim, tree, cfg.step_ms));
  else if (cfg.solver == CB_SOLVER_BE)
    p->eng.reset(make_be_io(host, stim, tree, cfg.step_ms));
  else
    p->eng.reset(make_global_io(host, sol, stim, poisson_of(cfg)));
  *out = p.release();
  return CB_OK;
}

// go_initialize + go_solve_initialize (go.cu:160-230, go_solve.cu:248-333):
// global FP64 engine only (the grid gap junctions couple the cells)
int create_go(const cb_pop_config &cfg, cb_pop **out) {
  const int n = cfg.nx * cfg.ny;
  if (n == 0) return fail(CB_E_ARG, "empty population");
  if (cfg.engine != CB_ENGINE_GLOBAL_FP64 && cfg.engine != CB_ENGINE_TREE_FP64)
    return fail(CB_E_UNSUP, "Golgi cells are gap-junction coupled: global engine only");
  GoHost host;
  std::string err;
  const std::string path = cfg.morph_path ? cfg.morph_path : "./Go_131.txt";
  if (!build_go_host(path, cfg.nx, cfg.ny, cfg.v0, host, err)) return fail(CB_E_IO, err);
  StimSpec stim;   // go_set_current (go.cu:258-268): the soma, [800, 1100) ms
  stim.comp = go::REC;
  stim.t0 = go::STIM_T0;
  stim.t1 = go::STIM_T1;
  if (cfg.stim_comp >= 0) {
    if (cfg.stim_comp >= go::COMP) return fail(CB_E_ARG, "stimulus compartment out of range");
    stim.comp = cfg.stim_comp;
    stim.t0 = cfg.stim_t0;
    stim.t1 = cfg.stim_t1;
  }
  stim.amp.assign(n, go::STIM);
  if (cfg.stim_amp)
    for (int c = 0; c < n; c++) stim.amp[c] = cfg.stim_amp[c];
  if (cfg.stim_comp == CB_STIM_NONE) stim.amp.assign(n, 0.0);
  SolverSpec sol;
  const double tol = 1.0e-6;   // TOL_GO, solve_rkc.cuh:29
  sol.atol = cfg.atol > 0 ? cfg.atol : tol;
  sol.rtol = cfg.rtol > 0 ? cfg.rtol : tol;
  sol.ion_interval = cfg.ion_interval_ms;
  sol.hmin = cfg.hmin_ms;
  sol.refresh_fn = cfg.refresh_fn != 0;
  if (cfg.rho_floor) return fail(CB_E_UNSUP, "the spectral-radius floor is provided for Purkinje cells");
  if (!(sol.atol > 0.0) || !(sol.rtol >= 0.0)) return fail(CB_E_ARG, "atol must be > 0 and rtol >= 0");
  std::unique_ptr<cb_pop> p(new cb_pop);
  p->cell_type = CB_GO;
  p->solver = cfg.solver;
  p->engine = cfg.engine;
  p->comp = go::COMP;
  p->device = cfg.device;
  CB_HIP(hipSetDevice(cfg.device));
  const bool tree = cfg.engine == CB_ENGINE_TREE_FP64;
  if (cfg.solver == CB_SOLVER_CN)
    p->eng.reset(make_cn_go(host, stim, tree, cfg.step_ms));
  else if (cfg.solver == CB_SOLVER_BE)
    p->eng.reset(make_be_go(host, stim, tree, cfg.step_ms));
  else
    p->eng.reset(make_global_go(host, sol, stim, poisson_of(cfg)));
  *out = p.release();
  return CB_OK;
}

// gr_initialize + gr_solve_initialize (gr.cu:151-218, gr_solve.cu:170-259):
// global FP64 engine (the reference's semantics)
int create_gr(const cb_pop_config &cfg, cb_pop **out) {
  const int n = cfg.nx * cfg.ny;
  if (n == 0) return fail(CB_E_ARG, "empty population");
  if (cfg.engine != CB_ENGINE_GLOBAL_FP64 && cfg.engine != CB_ENGINE_TREE_FP64)
    return fail(CB_E_UNSUP, "granule cells: global engine only");
  // a chain file (cb_synth_gr_chains) has comp rows per cell; Gr.txt 578
  const int comp = cfg.comp > 0 ? cfg.comp : gr::COMP;
  if (comp > gr::COMP) return fail(CB_E_ARG, "granule compartment count out of range");
  if (comp != gr::COMP && cfg.stim_comp == -1)
    return fail(CB_E_ARG, "a granule chain needs a stimulus compartment or CB_STIM_NONE");
  GrHost host;
  std::string err;
  const std::string path = cfg.morph_path ? cfg.morph_path : "./Gr.txt";
  if (!build_gr_host(path, cfg.nx, cfg.ny, cfg.v0, host, err, comp)) return fail(CB_E_IO, err);
  StimSpec stim;   // gr_set_current (gr.cu:245-254): compartment 16, [50, 100) ms
  stim.comp = gr::REC;
  stim.t0 = gr::STIM_T0;
  stim.t1 = gr::STIM_T1;
  if (cfg.stim_comp >= 0) {
    if (cfg.stim_comp >= comp) return fail(CB_E_ARG, "stimulus compartment out of range");
    stim.comp = cfg.stim_comp;
    stim.t0 = cfg.stim_t0;
    stim.t1 = cfg.stim_t1;
  }
  stim.amp.assign(n, gr::STIM);
  if (cfg.stim_amp)
    for (int c = 0; c < n; c++) stim.amp[c] = cfg.stim_amp[c];
  if (cfg.stim_comp == CB_STIM_NONE) {
    stim.amp.assign(n, 0.0);
    stim.comp = 0;
  }
  SolverSpec sol;
  const double tol = 1.0e-9;   // TOL_GR, solve_rkc.cuh:28
  sol.atol = cfg.atol > 0 ? cfg.atol : tol;
  sol.rtol = cfg.rtol > 0 ? cfg.rtol : tol;
  sol.ion_interval = cfg.ion_interval_ms;
  sol.hmin = cfg.hmin_ms;
  sol.refresh_fn = cfg.refresh_fn != 0;
  if (cfg.rho_floor) return fail(CB_E_UNSUP, "the spectral-radius floor is provided for Purkinje cells");
  if (!(sol.atol > 0.0) || !(sol.rtol >= 0.0)) return fail(CB_E_ARG, "atol must be > 0 and rtol >= 0");
  std::unique_ptr<cb_pop> p(new cb_pop);
  p->cell_type = CB_GR;
  p->solver = cfg.solver;
  p->engine = cfg.engine;
  p->comp = comp;
  p->device = cfg.device;
  CB_HIP(hipSetDevice(cfg.device));
  const bool tree = cfg.engine == CB_ENGINE_TREE_FP64;
  if (cfg.solver == CB_SOLVER_CN)
    p->eng.reset(make_cn_gr(host, stim, tree, cfg.step_ms));
  else if (cfg.solver == CB_SOLVER_BE)
    p->eng.reset(make_be_gr(host, stim, tree, cfg.step_ms));
  else
    p->eng.reset(make_global_gr(host, sol, stim, poisson_of(cfg)));
  *out = p.release();
  return CB_OK;
}

template <typename T>
T *dev_copy(const std::vector<T> &h) {
  void *p = nullptr;
  CB_HIP(hipMalloc(&p, sizeof(T) * (h.empty() ? 1 : h.size())));
  if (!h.empty()) CB_HIP(hipMemcpy(p, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
  return (T *)p;
}

// rebuilds the population's incoming-synapse CSR (entries of a compartment
// in set order, then synapse order) and hands it to the engine; the previous
// CSR is released only once the engine has taken the new one
void recouple(cb_pop *p) {
  CB_HIP(hipSetDevice(p->device));
  const int nn = p->eng->nc();
  SynIn in;
  int *row_d = nullptr, *slot_d = nullptr;
  if (!p->syn_in.empty()) {
    std::vector<int> row(nn + 1, 0);
    for (const cb_syn *s : p->syn_in)
      for (int k = 0; k < s->host.n; k++) row[s->host.post[k] + 1]++;
    for (int i = 0; i < nn; i++) row[i + 1] += row[i];
    std::vector<int> fill(row.begin(), row.end() - 1), slot(row[nn]);
    for (size_t t = 0; t < p->syn_in.size(); t++) {
      const cb_syn *s = p->syn_in[t];
      for (int k = 0; k < s->host.n; k++) slot[fill[s->host.post[k]]++] = (int)(t << 30) | k;
      in.val[t] = s->val_d;
      in.E[t] = s->host.E;
    }
    row_d = dev_copy(row);
    slot_d = dev_copy(slot);
    in.row = row_d;
    in.slot = slot_d;
  }
  p->eng->sync();
  try {
    p->eng->set_synapses(in);
  } catch (...) {
    if (row_d) (void)hipFree(row_d);
    if (slot_d) (void)hipFree(slot_d);
    throw;
  }
  if (p->syn_row) (void)hipFree(p->syn_row);
  if (p->syn_slot) (void)hipFree(p->syn_slot);
  p->syn_row = row_d;
  p->syn_slot = slot_d;
}

// creates a set from the host rules, uploads it and couples it into post
int make_syn(int kind, cb_pop *a, cb_pop *b, cb_pop *pre, cb_pop *post, const double *x1600, uint64_t seed,
             cb_syn **out) {
  std::unique_ptr<cb_syn> s(new cb_syn);
  const int nx_a = a ? a->nx : 0, ny_a = a ? a->ny : 0, nx_b = b ? b->nx : 0, ny_b = b ? b->ny : 0;
  build_syn(kind, nx_a, ny_a, nx_b, ny_b, x1600, seed, s->host);
  s->seed = seed;
  s->pre = pre;
  s->post = post;
  const int n = s->host.n;
  if (n > 0) {
    s->device = post->device;
    CB_HIP(hipSetDevice(s->device));
    s->pre_d = dev_copy(s->host.pre);
    s->w_d = dev_copy(s->host.weight);
    std::vector<double> zero(n, 0.0), thousand(n, 1000.0);
    for (int k = 0; k < 3; k++) s->x_d[k] = dev_copy(zero);
    s->val_d = dev_copy(zero);
    s->old_d = dev_copy(thousand);   // old_v = 1000: no spike on the first update
    // the reference couples every set except the inhibitory Purkinje input
    if (kind != SYN_MLIPKJ) {
      if (post->in_net) return fail(CB_E_UNSUP, "the population is coupled to a network");
      if (post->syn_in.size() >= 2) return fail(CB_E_UNSUP, "a population takes at most two synapse sets");
      post->syn_in.push_back(s.get());
      try {
        recouple(post);
      } catch (...) {
        post->syn_in.pop_back();
        throw;
      }
    }
  }
  *out = s.release();
  return CB_OK;
}

void syn_step(cb_syn *s, double t) {
  if (!s || s->host.n == 0) return;
  CB_HIP(hipSetDevice(s->device));
  const double *pv = nullptr;
  if (s->pre) {
    s->pre->eng->sync();
    s->pre->eng->check();
    pv = s->pre->eng->device_v();
    if (!pv) throw Error("the presynaptic population's engine exposes no voltage");
  }
  s->post->eng->sync();
  SynDev d{s->host.kind, s->host.n, s->pre_d, s->x_d[0], s->x_d[1], s->x_d[2], s->val_d, s->old_d, s->w_d,
           s->host.decay[0], s->host.decay[1], s->host.decay[2], (uint32_t)s->seed, (uint32_t)(s->seed >> 32)};
  hipStream_t st = s->post->eng->stream();
  syn_update(d, pv, t, s->step, st);
  CB_HIP(hipStreamSynchronize(st));
  s->step++;
}

bool read_location_x(const char *path, std::vector<double> &x, std::string &err) {
  std::FILE *f = std::fopen(path, "r");
  if (!f) {
    err = std::string("no such file ") + path;
    return false;
  }
  x.assign(1600, 0.0);
  for (int i = 0; i < 1600; i++) {
    int i1, i5;
    double i2, i3, i4;
    if (std::fscanf(f, "%d,%lf,%lf,%lf,%d", &i1, &i2, &i3, &i4, &i5) != 5) {
      std::fclose(f);
      err = std::string("PARAM_FILE_READING_ERROR in ") + path;
      return false;
    }
    x[i] = i2;
  }
  std::fclose(f);
  return true;
}

int solver_from_name(const char *s) {
  if (!s) return -1;
  if (std::strncmp(s, "BE", 2) == 0) return CB_SOLVER_BE;
  if (std::strncmp(s, "CN", 2) == 0) return CB_SOLVER_CN;
  if (std::strncmp(s, "RKC", 3) == 0) return CB_SOLVER_RKC;
  return -1;
}
}  // namespace

namespace {
NetSpec net_spec_of(const cb_net_config &c) {
  NetSpec s;
  s.seed = c.seed;
  s.deg[NET_MFGR] = c.deg_mf_gr;
  s.deg[NET_GOGR] = c.deg_go_gr;
  s.deg[NET_GRGO] = c.deg_gr_go;
  s.deg[NET_GRPKJ] = c.deg_gr_pkj;
  s.total = c.total;
  s.w_min_nS = c.w_min_nS;
  s.w_max_nS = c.w_max_nS;
  s.tau_ms[0] = c.tau_ampa_ms;
  s.tau_ms[1] = c.tau_gaba_ms;
  s.e_mV[0] = c.e_ampa_mV;
  s.e_mV[1] = c.e_gaba_mV;
  s.delay_ms = c.delay_ms;
  s.mf_rate_hz = c.mf_rate_hz;
  s.tgt_lo[NP_GR] = c.gr_target_comp;
  s.tgt_hi[NP_GR] = c.gr_target_comp + 1;
  s.tgt_lo[NP_GO] = c.go_target_lo;
  s.tgt_hi[NP_GO] = c.go_target_hi;
  s.tgt_lo[NP_PKJ] = c.pkj_target_lo;
  s.tgt_hi[NP_PKJ] = c.pkj_target_hi;
  s.spike_comp[NP_GR] = c.gr_spike_comp;
  s.spike_comp[NP_GO] = c.go_spike_comp;
  s.spike_comp[NP_PKJ] = c.pkj_spike_comp;
  s.thr_mV[NP_GR] = c.gr_thr_mV;
  s.thr_mV[NP_GO] = c.go_thr_mV;
  s.thr_mV[NP_PKJ] = c.pkj_thr_mV;
  return s;
}
}  // namespace

struct cb_net {
  std::unique_ptr<Network> net;
  cb_pop *pop[3] = {nullptr, nullptr, nullptr};
  int device = 0;
};

extern "C" {

const char *cb_last_error(void) { return g_err.c_str(); }

void cb_philox4x32_10(const uint32_t ctr[4], const uint32_t key[2], uint32_t out[4]) {
  u32x4 r = philox4x32_10(ctr[0], ctr[1], ctr[2], ctr[3], key[0], key[1]);
  for (int i = 0; i < 4; i++) out[i] = r.v[i];
}

int cb_config_default(cb_pop_config *cfg, int cell_type, int solver, int nx, int ny) {
  if (!cfg) return fail(CB_E_ARG, "null config");
  std::memset(cfg, 0, sizeof(*cfg));
  cfg->cell_type = cell_type;
  cfg->solver = solver;
  cfg->engine = CB_ENGINE_GLOBAL_FP64;
  cfg->nx = nx;
  cfg->ny = ny;
  cfg->atol = -1.0;
  cfg->rtol = -1.0;
  cfg->stim_comp = -1;
  cfg->poisson_rate_hz = 5.0;
  cfg->poisson_g_mS = 1e-6;
  cfg->poisson_tau_ms = 2.0;
  cfg->poisson_e_mV = 0.0;
  return CB_OK;
}

int cb_pop_create(const cb_pop_config *cfg, cb_pop **out) {
  const int rc = guarded([&]() -> int {
    if (!cfg || !out) return fail(CB_E_ARG, "null argument");
    *out = nullptr;
    if (cfg->nx < 0 || cfg->ny < 0) return fail(CB_E_ARG, "negative grid size");
    if (cfg->cell_type < CB_GR || cfg->cell_type > CB_IO) return fail(CB_E_ARG, "unknown cell type");
    if (cfg->solver != CB_SOLVER_RKC && cfg->solver != CB_SOLVER_CN && cfg->solver != CB_SOLVER_BE)
      return fail(CB_E_ARG, "unknown solver");
    if (cfg->solver != CB_SOLVER_RKC && cfg->engine != CB_ENGINE_GLOBAL_FP64 && cfg->engine != CB_ENGINE_TREE_FP64)
      return fail(CB_E_UNSUP, "the CN and BE solvers run on the global FP64 engine or the per-cell tree solve");
    if (cfg->solver == CB_SOLVER_RKC && cfg->engine == CB_ENGINE_TREE_FP64)
      return fail(CB_E_UNSUP, "the per-cell tree solve is provided for the CN and BE solvers");
    if (cfg->solver == CB_SOLVER_RKC && cfg->step_ms > 0.0)
      return fail(CB_E_ARG, "step_ms applies to the CN and BE solvers (RKC chooses its own steps)");
    if (cfg->hmin_ms > 0.125) return fail(CB_E_ARG, "hmin_ms must not exceed H_MAX = 0.125 ms");
    if (cfg->comp > 0 && cfg->cell_type != CB_GR)
      return fail(CB_E_ARG, "comp applies to granule chains (the other formats fix the compartment count)");
    if (cfg->solver != CB_SOLVER_RKC && cfg->poisson_on)
      return fail(CB_E_UNSUP, "the Poisson conductance drive is provided for the RKC solver");
    // the device is selected right before an engine is built, so argument
    // and file errors are reported without touching a GPU
    if (cfg->cell_type == CB_IO) return create_io(*cfg, out);
    if (cfg->cell_type == CB_GO) return create_go(*cfg, out);
    if (cfg->cell_type == CB_GR) return create_gr(*cfg, out);
    std::vector<MorphRow> rows;
    std::string err;
    const std::string mpath = cfg->morph_path ? cfg->morph_path : "./Pkj.txt";
    if (!read_pkj_morph(mpath, pkj::COMP, rows, err)) return fail(CB_E_IO, err);
    std::vector<int> gpre, gpost;
    const int n = cfg->nx * cfg->ny;
    if (n == 0) return fail(CB_E_ARG, "empty population");
    // a grid reads its gap-junction pairs from ./Pkj_GJ.csv unless told
    // otherwise, and a missing file is an error as in pkj_solve.cu:86-87;
    // gj_path = "" asks for uncoupled cells
    bool use_gj = n > 1 && !(cfg->gj_path && cfg->gj_path[0] == '\0');
    if (use_gj) {
      const std::string gpath = cfg->gj_path ? cfg->gj_path : "./Pkj_GJ.csv";
      if (!read_pkj_gj(gpath, gpre, gpost, err)) return fail(CB_E_IO, err);
    }
    PkjHost host;
    if (!build_pkj_host(rows, cfg->nx, cfg->ny, use_gj ? &gpre : nullptr, use_gj ? &gpost : nullptr, cfg->v0, host,
                        err))
      return fail(CB_E_IO, err);
    StimSpec stim;
    if (cfg->stim_comp >= 0) {
      if (cfg->stim_comp >= pkj::COMP) return fail(CB_E_ARG, "stimulus compartment out of range");
      stim.comp = cfg->stim_comp;
      stim.t0 = cfg->stim_t0;
      stim.t1 = cfg->stim_t1;
    }
    stim.amp.assign(n, pkj::CURRENT);
    if (cfg->stim_amp)
      for (int c = 0; c < n; c++) stim.amp[c] = cfg->stim_amp[c];
    if (cfg->stim_comp == CB_STIM_NONE) stim.amp.assign(n, 0.0);
    PoissonSpec syn;
    syn.on = cfg->poisson_on != 0;
    syn.rate_hz = cfg->poisson_rate_hz;
    syn.g_event = cfg->poisson_g_mS;
    syn.tau_ms = cfg->poisson_tau_ms;
    syn.e_syn = cfg->poisson_e_mV;
    syn.seed = cfg->poisson_seed;
    const double tol = 1.0e-6;   // TOL_PKJ, solve_rkc.cuh:29
    SolverSpec sol;
    sol.atol = cfg->atol > 0 ? cfg->atol : tol;
    sol.rtol = cfg->rtol > 0 ? cfg->rtol : tol;
    sol.ion_interval = cfg->ion_interval_ms;
    sol.hmin = cfg->hmin_ms;
    sol.refresh_fn = cfg->refresh_fn != 0;
    if (cfg->rho_floor) {
      std::vector<double> rho;
      cable_spectral_radius(host, rho);
      sol.rho_floor.resize(rho.size());
      for (size_t c = 0; c < rho.size(); c++) sol.rho_floor[c] = 1.2 * rho[c];
    }
    // atol > 0 keeps every error weight positive (the reference asserts on a
    // zero weight, idid = 3, solve_rkc.cu:50-53)
    if (!(sol.atol > 0.0) || !(sol.rtol >= 0.0)) return fail(CB_E_ARG, "atol must be > 0 and rtol >= 0");
    std::unique_ptr<cb_pop> p(new cb_pop);
    p->cell_type = cfg->cell_type;
    p->solver = cfg->solver;
    p->engine = cfg->engine;
    p->comp = pkj::COMP;
    p->device = cfg->device;
    if (cfg->solver == CB_SOLVER_RKC &&
        (cfg->engine == CB_ENGINE_CELL_FP64 || cfg->engine == CB_ENGINE_CELL_MIXED) && host.n_gj > 0)
      return fail(CB_E_UNSUP, "per-cell engines need cells without intercell gap junctions");
    CB_HIP(hipSetDevice(cfg->device));
    if (cfg->solver != CB_SOLVER_RKC) {
      const bool tree = cfg->engine == CB_ENGINE_TREE_FP64;
      p->eng.reset(cfg->solver == CB_SOLVER_CN ? make_cn_pkj(host, stim, tree, cfg->step_ms)
                                               : make_be_pkj(host, stim, tree, cfg->step_ms));
      *out = p.release();
      return CB_OK;
    }
    switch (cfg->engine) {
      case CB_ENGINE_GLOBAL_FP64:
        p->eng.reset(make_global_pkj(host, sol, stim, syn));
        break;
      case CB_ENGINE_CELL_FP64:
      case CB_ENGINE_CELL_MIXED:
        p->eng.reset(make_cell_pkj(host, sol, stim, syn, cfg->engine == CB_ENGINE_CELL_MIXED));
        break;
      default:
        return fail(CB_E_ARG, "unknown engine");
    }
    *out = p.release();
    return CB_OK;
  });
  if (rc == CB_OK && out && *out) {
    (*out)->nx = cfg->nx;
    (*out)->ny = cfg->ny;
  }
  return rc;
}

int cb_pop_destroy(cb_pop *p) {
  return guarded([&]() -> int {
    if (!p) return CB_OK;
    if (p->in_net) return fail(CB_E_ARG, "the population is coupled to a network: destroy the network first");
    CB_HIP(hipSetDevice(p->device));
    delete p;
    return CB_OK;
  });
}

int cb_pop_set_current(cb_pop *p, double t) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    p->eng->set_current(t);
    return CB_OK;
  });
}

int cb_pop_advance(cb_pop *p) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    p->eng->advance();
    return CB_OK;
  });
}

int cb_pop_run(cb_pop *p, int nsteps, double t0, int rec_comp, double *rec_out) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (nsteps < 0) return fail(CB_E_ARG, "negative step count");
    if (rec_out && (rec_comp < CB_REC_ALL || rec_comp >= p->comp))
      return fail(CB_E_ARG, "record compartment out of range");
    p->eng->run(nsteps, t0, rec_comp, rec_out);
    return CB_OK;
  });
}

int cb_pop_set_raster(cb_pop *p, int comp, double thr) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (comp >= p->comp) return fail(CB_E_ARG, "raster compartment out of range");
    p->eng->set_raster(comp, thr);
    return CB_OK;
  });
}

int cb_pop_spikes(cb_pop *p, int cap, double *t_out, int *cell_out, int *n_out) {
  return guarded([&]() -> int {
    if (!p || !n_out || (cap > 0 && (!t_out || !cell_out))) return fail(CB_E_ARG, "null argument");
    *n_out = p->eng->take_spikes(cap, t_out, cell_out);
    return CB_OK;
  });
}

int cb_pop_run_noalloc(cb_pop *p, int nsteps, double t0, int rec_comp, double *rec_out) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (nsteps < 0) return fail(CB_E_ARG, "negative step count");
    if (rec_out && (rec_comp < 0 || rec_comp >= p->comp)) return fail(CB_E_ARG, "record compartment out of range");
    CB_HIP(hipSetDevice(p->device));
    p->eng->run_noalloc(nsteps, t0, rec_comp, rec_out);
    return CB_OK;
  });
}

int cb_pop_read(cb_pop *p, int field, double *dst) {
  return guarded([&]() -> int {
    if (!p || !dst) return fail(CB_E_ARG, "null argument");
    p->eng->read(field, dst);
    return CB_OK;
  });
}

int cb_pop_size(const cb_pop *p, int *ncell, int *nc) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (ncell) *ncell = p->eng->ncell();
    if (nc) *nc = p->eng->nc();
    return CB_OK;
  });
}

int cb_pop_stats(const cb_pop *p, int64_t *out6) {
  return guarded([&]() -> int {
    if (!p || !out6) return fail(CB_E_ARG, "null argument");
    Stats s = p->eng->stats();
    out6[0] = s.steps;
    out6[1] = s.rejects;
    out6[2] = s.stages;
    out6[3] = s.rho_iters;
    out6[4] = s.ion_updates;
    out6[5] = s.macro_steps;
    return CB_OK;
  });
}

int cb_pop_kernel_time(cb_pop *p, double *ms, int64_t *launches, int reset) {
  return guarded([&]() -> int {
    if (!p || !ms || !launches) return fail(CB_E_ARG, "null argument");
    long n = 0;
    p->eng->kernel_time(ms, &n, reset != 0);
    *launches = n;
    return CB_OK;
  });
}

int cb_pop_autotune(cb_pop *p, int trial_steps, int *threads) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (threads && *threads > 0) {
      if (!p->eng->select_mapping(*threads)) return fail(CB_E_ARG, "no such mapping");
      return CB_OK;
    }
    int t = p->eng->autotune(trial_steps, -1.0);   // trial from the current time
    if (threads) *threads = t;
    return CB_OK;
  });
}

int cb_pop_mapping(const cb_pop *p, char *buf, int len) {
  return guarded([&]() -> int {
    if (!p || !buf || len <= 0) return fail(CB_E_ARG, "null argument");
    const std::string m = p->eng->mapping();
    std::snprintf(buf, (size_t)len, "%s", m.c_str());
    return (int)m.size() < len ? CB_OK : fail(CB_E_ARG, "buffer too short for the mapping description");
  });
}

int cb_pop_launch_path(cb_pop *p, int on) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (!p->eng->use_launches(on != 0)) return fail(CB_E_UNSUP, "the population has one path only");
    return CB_OK;
  });
}

int cb_pop_wait_limit(cb_pop *p, double seconds) {
  return guarded([&]() -> int {
    if (!p) return fail(CB_E_ARG, "null population");
    if (!(seconds >= 0.0) || seconds > 1e9) return fail(CB_E_ARG, "the limit must be 0 to 1e9 s");
    p->eng->wait_limit(seconds);
    return CB_OK;
  });
}

int cb_pop_controller(const cb_pop *p, double *o, double *hw) {
  return guarded([&]() -> int {
    if (!p || !o || !hw) return fail(CB_E_ARG, "null argument");
    if (p->engine != CB_ENGINE_GLOBAL_FP64) return fail(CB_E_UNSUP, "per-cell engines have no global controller");
    p->eng->controller(o, hw);
    return CB_OK;
  });
}

int cb_synth_pkj_morph(const char *path, uint64_t seed, int ncell, double soma_r_um, double lmin_um, double lmax_um,
                       double d0_um, double d1_um, const double *dscale) {
  return guarded([&]() -> int {
    if (!path || ncell <= 0) return fail(CB_E_ARG, "bad argument");
    if (!(lmin_um > 0) || lmax_um < lmin_um || !(d1_um > 0) || !(d0_um > 0) || !(soma_r_um > 0))
      return fail(CB_E_ARG, "bad geometry");
    std::vector<MorphRow> all, one;
    all.reserve((size_t)ncell * pkj::COMP);
    for (int c = 0; c < ncell; c++) {
      synth_pkj_tree(seed + (uint64_t)c, pkj::COMP, soma_r_um, lmin_um, lmax_um, d0_um, d1_um, dscale ? dscale[c] : 1.0,
                     one);
      all.insert(all.end(), one.begin(), one.end());
    }
    std::string err;
    if (!write_pkj_morph(path, all, err)) return fail(CB_E_IO, err);
    return CB_OK;
  });
}

int cb_pkj_cable_spectral_radius(const char *morph_path, int ncell, double *rho) {
  return guarded([&]() -> int {
    if (!morph_path || !rho || ncell <= 0) return fail(CB_E_ARG, "bad argument");
    std::vector<MorphRow> rows;
    std::string err;
    if (!read_pkj_morph(morph_path, pkj::COMP, rows, err)) return fail(CB_E_IO, err);
    std::vector<double> v0(ncell, pkj::V_INIT);
    PkjHost host;
    if (!build_pkj_host(rows, ncell, 1, nullptr, nullptr, v0.data(), host, err)) return fail(CB_E_IO, err);
    std::vector<double> r;
    cable_spectral_radius(host, r);
    for (int c = 0; c < ncell; c++) rho[c] = r[c];
    return CB_OK;
  });
}

int cb_pkj_initialize(int nx, int ny, const char *solver, cb_pop **out) {
  int s = solver_from_name(solver);
  if (s < 0) return fail(CB_E_ARG, "error in pkj_initialize: unknown solver");
  cb_pop_config cfg;
  cb_config_default(&cfg, CB_PKJ, s, nx, ny);
  return cb_pop_create(&cfg, out);
}

int cb_io_initialize(int nx, int ny, const char *solver, cb_pop **out) {
  int s = solver_from_name(solver);
  if (s < 0) return fail(CB_E_ARG, "error in io_initialize");
  cb_pop_config cfg;
  cb_config_default(&cfg, CB_IO, s, nx, ny);
  return cb_pop_create(&cfg, out);
}

int cb_io_solve_update_v(cb_pop *p) { return cb_pop_advance(p); }
int cb_io_set_current(cb_pop *p, double t) { return cb_pop_set_current(p, t); }
int cb_io_finalize(cb_pop *p) { return cb_pop_destroy(p); }

int cb_io_output_file(const cb_pop *p, const double *memv, double *raster_prev, double t, const char *v_csv,
                      const char *raster_csv) {
  if (!p || !memv || !raster_prev) return fail(CB_E_ARG, "null argument");
  if (p->cell_type != CB_IO) return fail(CB_E_ARG, "not an inferior-olive population");
  const int n = p->eng->ncell(), C = p->comp;
  if (v_csv) {
    FILE *f = std::fopen(v_csv, "a");
    if (!f) return fail(CB_E_IO, std::string("cannot open ") + v_csv);
    std::fprintf(f, "%lf,", t);
    for (int j = 0; j < n; j++)
      for (int k = 0; k < C; k++) std::fprintf(f, "%lf,", memv[k + (size_t)j * C]);
    std::fprintf(f, "\n");
    std::fclose(f);
  }
  FILE *fr = raster_csv ? std::fopen(raster_csv, "a") : nullptr;
  if (raster_csv && !fr) return fail(CB_E_IO, std::string("cannot open ") + raster_csv);
  for (int j = 0; j < n; j++) {
    const double vj = memv[2 + (size_t)j * C];
    if (vj > 10.0 && raster_prev[j] <= 10.0 && fr) std::fprintf(fr, "%lf,%d\n", t, j);
    raster_prev[j] = vj;
  }
  if (fr) std::fclose(fr);
  return CB_OK;
}

int cb_gr_initialize(int nx, int ny, const char *solver, cb_pop **out) {
  int s = solver_from_name(solver);
  if (s < 0) return fail(CB_E_ARG, "error in gr_initialize");
  cb_pop_config cfg;
  cb_config_default(&cfg, CB_GR, s, nx, ny);
  return cb_pop_create(&cfg, out);
}

int cb_gr_solve_update_v(cb_pop *p) { return cb_pop_advance(p); }
int cb_gr_set_current(cb_pop *p, double t) { return cb_pop_set_current(p, t); }
int cb_gr_finalize(cb_pop *p) { return cb_pop_destroy(p); }

int cb_gr_output_file(const cb_pop *p, const double *memv, double *raster_prev, double t, const char *v_csv,
                      const char *raster_csv) {
  if (!p || !memv || !raster_prev) return fail(CB_E_ARG, "null argument");
  if (p->cell_type != CB_GR) return fail(CB_E_ARG, "not a granule-cell population");
  const int n = p->eng->ncell(), C = p->comp;
  if (v_csv) {
    FILE *f = std::fopen(v_csv, "a");
    if (!f) return fail(CB_E_IO, std::string("cannot open ") + v_csv);
    std::fprintf(f, "%lf,", t);
    for (int j = 0; j < n; j++) std::fprintf(f, "%lf,", memv[gr::REC + (size_t)j * C]);
    std::fprintf(f, "\n");
    std::fclose(f);
  }
  FILE *fr = raster_csv ? std::fopen(raster_csv, "a") : nullptr;
  if (raster_csv && !fr) return fail(CB_E_IO, std::string("cannot open ") + raster_csv);
  for (int j = 0; j < n; j++) {
    const double vj = memv[gr::RASTER + (size_t)j * C];
    if (vj > 10.0 && raster_prev[j] <= 10.0 && fr) std::fprintf(fr, "%lf,%d\n", t, j);
    raster_prev[j] = vj;
  }
  if (fr) std::fclose(fr);
  return CB_OK;
}

int cb_go_initialize(int nx, int ny, const char *solver, cb_pop **out) {
  int s = solver_from_name(solver);
  if (s < 0) return fail(CB_E_ARG, "error in go_initialize");
  cb_pop_config cfg;
  cb_config_default(&cfg, CB_GO, s, nx, ny);
  return cb_pop_create(&cfg, out);
}

int cb_go_solve_update_v(cb_pop *p) { return cb_pop_advance(p); }
int cb_go_set_current(cb_pop *p, double t) { return cb_pop_set_current(p, t); }
int cb_go_finalize(cb_pop *p) { return cb_pop_destroy(p); }

int cb_go_output_file(const cb_pop *p, const double *memv, double *raster_prev, double t, const char *v_csv,
                      const char *raster_csv) {
  if (!p || !memv || !raster_prev) return fail(CB_E_ARG, "null argument");
  if (p->cell_type != CB_GO) return fail(CB_E_ARG, "not a Golgi-cell population");
  const int n = p->eng->ncell(), C = p->comp;
  if (v_csv) {
    FILE *f = std::fopen(v_csv, "a");
    if (!f) return fail(CB_E_IO, std::string("cannot open ") + v_csv);
    std::fprintf(f, "%lf,", t);
    for (int j = 0; j < n; j++) std::fprintf(f, "%lf,", memv[go::REC + (size_t)j * C]);
    std::fprintf(f, "\n");
    std::fclose(f);
  }
  FILE *fr = raster_csv ? std::fopen(raster_csv, "a") : nullptr;
  if (raster_csv && !fr) return fail(CB_E_IO, std::string("cannot open ") + raster_csv);
  for (int j = 0; j < n; j++) {
    const double vj = memv[go::REC + (size_t)j * C];
    if (vj > 10.0 && raster_prev[j] <= 10.0 && fr) std::fprintf(fr, "%lf,%d\n", t, j);
    raster_prev[j] = vj;
  }
  if (fr) std::fclose(fr);
  return CB_OK;
}

int cb_pkj_solve_update_v(cb_pop *p) { return cb_pop_advance(p); }
int cb_pkj_set_current(cb_pop *p, double t) { return cb_pop_set_current(p, t); }
int cb_pkj_finalize(cb_pop *p) { return cb_pop_destroy(p); }

int cb_pkj_output_file(const cb_pop *p, const double *memv, double *raster_prev, double t, const char *v_csv,
                       const char *raster_csv) {
  if (!p || !memv || !raster_prev) return fail(CB_E_ARG, "null argument");
  const int n = p->eng->ncell(), C = p->comp;
  if (v_csv) {
    FILE *f = std::fopen(v_csv, "a");
    if (!f) return fail(CB_E_IO, std::string("cannot open ") + v_csv);
    std::fprintf(f, "%lf,", t);
    for (int j = 0; j < n; j++) std::fprintf(f, "%lf,", memv[1599 + (size_t)j * C]);
    std::fprintf(f, "\n");
    std::fclose(f);
  }
  FILE *fr = raster_csv ? std::fopen(raster_csv, "a") : nullptr;
  if (raster_csv && !fr) return fail(CB_E_IO, std::string("cannot open ") + raster_csv);
  for (int j = 0; j < n; j++) {
    double vj = memv[1599 + (size_t)j * C];
    if (vj > -10.0 && raster_prev[j] <= -10.0 && fr) std::fprintf(fr, "%lf,%d\n", t, j);
    raster_prev[j] = vj;
  }
  if (fr) std::fclose(fr);
  return CB_OK;
}


int cb_mfgr_create(cb_pop *gr, uint64_t seed, cb_syn **out) {
  return guarded([&]() -> int {
    if (!out) return fail(CB_E_ARG, "null argument");
    if (gr && gr->cell_type != CB_GR) return fail(CB_E_ARG, "mfgr_create takes a granule population");
    return make_syn(SYN_MFGR, gr, nullptr, nullptr, gr, nullptr, seed, out);
  });
}

int cb_gogr_create(cb_pop *go, cb_pop *gr, cb_syn **out) {
  return guarded([&]() -> int {
    if (!out) return fail(CB_E_ARG, "null argument");
    if ((go && go->cell_type != CB_GO) || (gr && gr->cell_type != CB_GR))
      return fail(CB_E_ARG, "gogr_create takes a Golgi and a granule population");
    return make_syn(SYN_GOGR, go, gr, go, gr, nullptr, 0, out);
  });
}

int cb_grgo_create(cb_pop *gr, cb_pop *go, cb_syn **out) {
  return guarded([&]() -> int {
    if (!out) return fail(CB_E_ARG, "null argument");
    if ((go && go->cell_type != CB_GO) || (gr && gr->cell_type != CB_GR))
      return fail(CB_E_ARG, "grgo_create takes a granule and a Golgi population");
    return make_syn(SYN_GRGO, gr, go, gr, go, nullptr, 0, out);
  });
}

int cb_grpkj_create(cb_pop *gr, cb_pop *pkj, const char *location_csv, uint64_t seed, cb_syn **out) {
  return guarded([&]() -> int {
    if (!out) return fail(CB_E_ARG, "null argument");
    if ((gr && gr->cell_type != CB_GR) || (pkj && pkj->cell_type != CB_PKJ))
      return fail(CB_E_ARG, "grpkj_create takes a granule and a Purkinje population");
    std::vector<double> x;
    if (gr && pkj && gr->nx * gr->ny > 0 && pkj->nx * pkj->ny > 0) {
      std::string err;
      if (!read_location_x(location_csv ? location_csv : "./Pkj_location_info.csv", x, err))
        return fail(CB_E_IO, err);
    }
    return make_syn(SYN_GRPKJ, gr, pkj, gr, pkj, x.empty() ? nullptr : x.data(), seed, out);
  });
}

int cb_mlipkj_create(cb_pop *pkj, cb_pop *gr, uint64_t seed, cb_syn **out) {
  return guarded([&]() -> int {
    if (!out) return fail(CB_E_ARG, "null argument");
    if ((gr && gr->cell_type != CB_GR) || (pkj && pkj->cell_type != CB_PKJ))
      return fail(CB_E_ARG, "mlipkj_create takes a Purkinje and a granule population");
    return make_syn(SYN_MLIPKJ, pkj, gr, nullptr, pkj, nullptr, seed, out);
  });
}

int cb_syn_finalize(cb_syn *s) {
  return guarded([&]() -> int {
    if (!s) return CB_OK;
    std::unique_ptr<cb_syn> own(s);
    if (s->post) {
      auto &v = s->post->syn_in;
      for (size_t t = 0; t < v.size(); t++)
        if (v[t] == s) {
          v.erase(v.begin() + t);
          recouple(s->post);
          break;
        }
    }
    if (s->host.n > 0) CB_HIP(hipSetDevice(s->device));
    return CB_OK;
  });
}

int cb_gr_synapse_update(double t, cb_syn *mfgr, cb_syn *gogr) {
  return guarded([&]() -> int {
    syn_step(mfgr, t);
    syn_step(gogr, t);
    return CB_OK;
  });
}

int cb_go_synapse_update(double t, cb_syn *grgo) {
  return guarded([&]() -> int {
    syn_step(grgo, t);
    return CB_OK;
  });
}

int cb_pkj_synapse_update(double t, cb_syn *grpkj, cb_syn *mlipkj) {
  (void)mlipkj;   // mlipkj_update is commented out in every branch of pkj_synapse_update
  return guarded([&]() -> int {
    syn_step(grpkj, t);
    return CB_OK;
  });
}

int cb_syn_size(const cb_syn *s, int *n) {
  if (!s || !n) return fail(CB_E_ARG, "null argument");
  *n = s->host.n;
  return CB_OK;
}

int cb_syn_comp(const cb_syn *s, int *pre, int *post) {
  if (!s || !pre || !post) return fail(CB_E_ARG, "null argument");
  std::memcpy(pre, s->host.pre.data(), sizeof(int) * s->host.n);
  std::memcpy(post, s->host.post.data(), sizeof(int) * s->host.n);
  return CB_OK;
}

int cb_syn_read(const cb_syn *s, int field, double *dst) {
  return guarded([&]() -> int {
    if (!s || !dst) return fail(CB_E_ARG, "null argument");
    if (s->host.n == 0) return CB_OK;
    const double *src = nullptr;
    switch (field) {
      case CB_SYN_TRACE0: case CB_SYN_TRACE1: case CB_SYN_TRACE2: src = s->x_d[field]; break;
      case CB_SYN_WEIGHT: src = s->w_d; break;
      case CB_SYN_VAL: src = s->val_d; break;
      case CB_SYN_OLD_V: src = s->old_d; break;
      default: return fail(CB_E_ARG, "unknown synapse field");
    }
    CB_HIP(hipSetDevice(s->device));
    if (s->post) s->post->eng->sync();
    CB_HIP(hipMemcpy(dst, src, sizeof(double) * s->host.n, hipMemcpyDeviceToHost));
    return CB_OK;
  });
}

int cb_syn_build(int kind, int nx_a, int ny_a, int nx_b, int ny_b, const double *x1600, uint64_t seed, int *n,
                 int *pre, int *post, double *weight) {
  return guarded([&]() -> int {
    if (!n) return fail(CB_E_ARG, "null argument");
    if (kind < CB_SYN_MFGR || kind > CB_SYN_MLIPKJ) return fail(CB_E_ARG, "unknown synapse kind");
    if (nx_a < 0 || ny_a < 0 || nx_b < 0 || ny_b < 0) return fail(CB_E_ARG, "negative grid size");
    if (kind == CB_SYN_GRPKJ && nx_a * ny_a > 0 && nx_b * ny_b > 0 && !x1600)
      return fail(CB_E_ARG, "the granule-Purkinje rule needs the compartment x positions");
    SynHost h;
    build_syn(kind, nx_a, ny_a, nx_b, ny_b, x1600, seed, h);
    *n = h.n;
    if (pre && post && weight) {
      std::memcpy(pre, h.pre.data(), sizeof(int) * h.n);
      std::memcpy(post, h.post.data(), sizeof(int) * h.n);
      std::memcpy(weight, h.weight.data(), sizeof(double) * h.n);
    }
    return CB_OK;
  });
}

struct cb_mix {
  std::unique_ptr<Mix> m;
  int device = 0;
};

// cb_mix_create validates its configuration and then refuses while this is
// set (see there)
constexpr bool mix_engine_switched_off = true;

int cb_mix_config_default(cb_mix_config *cfg) {
  if (!cfg) return fail(CB_E_ARG, "null config");
  std::memset(cfg, 0, sizeof(*cfg));
  cfg->interval_ms = 0.125;
  cfg->pkj_atol = 1e-6;
  cfg->pkj_rtol = 1e-6;
  cfg->pkj_stable = 1;
  cfg->pop[CB_GR].comp = 4;
  cfg->pop[CB_GR].stim_comp = 1;
  cfg->pop[CB_GR].rec_comp = 3;
  cfg->pop[CB_GR].thr = 10.0;
  cfg->pop[CB_GO].stim_comp = 30;
  cfg->pop[CB_GO].rec_comp = 30;
  cfg->pop[CB_GO].thr = 10.0;
  cfg->pop[CB_PKJ].stim_comp = 1599;
  cfg->pop[CB_PKJ].rec_comp = 1599;
  cfg->pop[CB_PKJ].thr = -10.0;
  cfg->pop[CB_IO].stim_comp = 0;
  cfg->pop[CB_IO].rec_comp = 2;
  cfg->pop[CB_IO].thr = 10.0;
  return CB_OK;
}

int cb_mix_create(const cb_mix_config *cfg, cb_mix **out) {
  return guarded([&]() -> int {
    if (!cfg || !out) return fail(CB_E_ARG, "null argument");
    *out = nullptr;
    MixSpec S;
    for (int t = 0; t < 4; t++) {
      const cb_mix_pop &q = cfg->pop[t];
      if (q.n < 0) return fail(CB_E_ARG, "negative cell count");
      if (q.n == 0) continue;
      if (!q.morph_path || !q.v0) return fail(CB_E_ARG, "a population needs a morphology file and initial voltages");
      MixPopSpec &p = S.pop[t];
      p.n = q.n;
      p.morph = q.morph_path;
      p.comp = q.comp;
      p.v0.assign(q.v0, q.v0 + q.n);
      if (q.amp) p.amp.assign(q.amp, q.amp + q.n);
      p.stim_comp = q.stim_comp;
      p.rec_comp = q.rec_comp;
      p.thr = q.thr;
      std::FILE *f = std::fopen(q.morph_path, "r");
      if (!f) return fail(CB_E_IO, std::string("no such file ") + q.morph_path);
      std::fclose(f);
    }
    if (cfg->pop[CB_PKJ].n > 0 &&
        (cfg->pop[CB_PKJ].stim_comp < 0 || cfg->pop[CB_PKJ].stim_comp >= pkj::COMP ||
         cfg->pop[CB_PKJ].rec_comp < 0 || cfg->pop[CB_PKJ].rec_comp >= pkj::COMP))
      return fail(CB_E_ARG, "Purkinje stimulated or recorded compartment out of range");
    if (cfg->io_gj_path) S.io_gj = cfg->io_gj_path;
    S.interval = cfg->interval_ms > 0 ? cfg->interval_ms : 0.125;
    S.pkj_atol = cfg->pkj_atol > 0 ? cfg->pkj_atol : 1e-6;
    S.pkj_rtol = cfg->pkj_rtol > 0 ? cfg->pkj_rtol : 1e-6;
    S.pkj_stable = cfg->pkj_stable != 0;
    // The batched engine is switched off: the first device run of its tests
    // ended with a GPU memory fault whose cause has not been found (the
    // small-cell body is in bounds in a host emulation of the same source).
    // It stays off until that cause is shown and fixed.
    if (mix_engine_switched_off)
      return fail(CB_E_UNSUP, "the batched mix engine is switched off: its first GPU run faulted and the cause "
                              "has not been found");
    CB_HIP(hipSetDevice(cfg->device));
    std::unique_ptr<cb_mix> m(new cb_mix);
    m->device = cfg->device;
    m->m.reset(make_mix(S));
    *out = m.release();
    return CB_OK;
  });
}

int cb_mix_run(cb_mix *m, int nint, double *rec_out, uint32_t *spk_out) {
  return guarded([&]() -> int {
    if (!m) return fail(CB_E_ARG, "null mix");
    if (nint < 0) return fail(CB_E_ARG, "negative interval count");
    CB_HIP(hipSetDevice(m->device));
    m->m->run(nint, rec_out, spk_out);
    return CB_OK;
  });
}

int cb_mix_layout(const cb_mix *m, int *ncell4, int *word_off4, int *words, int *lanes4) {
  return guarded([&]() -> int {
    if (!m) return fail(CB_E_ARG, "null mix");
    for (int t = 0; t < 4; t++) {
      if (ncell4) ncell4[t] = m->m->ncell(t);
      if (word_off4) word_off4[t] = m->m->word_off(t);
      if (lanes4) lanes4[t] = m->m->lanes(t);
    }
    if (words) *words = m->m->words();
    return CB_OK;
  });
}

int cb_mix_stats(const cb_mix *m, int type, int64_t *out6) {
  return guarded([&]() -> int {
    if (!m || !out6) return fail(CB_E_ARG, "null argument");
    if (type < 0 || type > 3) return fail(CB_E_ARG, "unknown cell type");
    const Stats s = m->m->stats(type);
    out6[0] = s.steps;
    out6[1] = s.rejects;
    out6[2] = s.stages;
    out6[3] = s.rho_iters;
    out6[4] = s.ion_updates;
    out6[5] = s.macro_steps;
    return CB_OK;
  });
}

int cb_mix_autotune(cb_mix *m, int trial_intervals, int *lanes4) {
  return guarded([&]() -> int {
    if (!m) return fail(CB_E_ARG, "null mix");
    CB_HIP(hipSetDevice(m->device));
    m->m->autotune(trial_intervals);
    if (lanes4)
      for (int t = 0; t < 4; t++) lanes4[t] = m->m->lanes(t);
    return CB_OK;
  });
}

int cb_mix_kernel_time(cb_mix *m, double *ms, int64_t *launches, int reset) {
  return guarded([&]() -> int {
    if (!m || !ms || !launches) return fail(CB_E_ARG, "null argument");
    long n = 0;
    m->m->kernel_time(ms, &n, reset != 0);
    *launches = n;
    return CB_OK;
  });
}

int cb_mix_use_graph(cb_mix *m, int on) {
  return guarded([&]() -> int {
    if (!m) return fail(CB_E_ARG, "null mix");
    m->m->use_graph(on != 0);
    return CB_OK;
  });
}

int cb_mix_destroy(cb_mix *m) {
  return guarded([&]() -> int {
    if (!m) return CB_OK;
    CB_HIP(hipSetDevice(m->device));
    delete m;
    return CB_OK;
  });
}

int cb_net_config_default(cb_net_config *cfg) {
  return guarded([&]() -> int {
    if (!cfg) return fail(CB_E_ARG, "null config");
    std::memset(cfg, 0, sizeof(*cfg));
    const NetSpec s;
    cfg->seed = s.seed;
    cfg->deg_mf_gr = s.deg[NET_MFGR];
    cfg->deg_go_gr = s.deg[NET_GOGR];
    cfg->deg_gr_go = s.deg[NET_GRGO];
    cfg->deg_gr_pkj = s.deg[NET_GRPKJ];
    cfg->total = s.total;
    cfg->w_min_nS = s.w_min_nS;
    cfg->w_max_nS = s.w_max_nS;
    cfg->tau_ampa_ms = s.tau_ms[0];
    cfg->tau_gaba_ms = s.tau_ms[1];
    cfg->e_ampa_mV = s.e_mV[0];
    cfg->e_gaba_mV = s.e_mV[1];
    cfg->delay_ms = s.delay_ms;
    cfg->mf_rate_hz = s.mf_rate_hz;
    cfg->gr_target_comp = 0;
    cfg->go_target_lo = s.tgt_lo[NP_GO];
    cfg->go_target_hi = s.tgt_hi[NP_GO];
    cfg->pkj_target_lo = s.tgt_lo[NP_PKJ];
    cfg->pkj_target_hi = s.tgt_hi[NP_PKJ];
    cfg->gr_spike_comp = s.spike_comp[NP_GR];
    cfg->go_spike_comp = s.spike_comp[NP_GO];
    cfg->pkj_spike_comp = s.spike_comp[NP_PKJ];
    cfg->gr_thr_mV = s.thr_mV[NP_GR];
    cfg->go_thr_mV = s.thr_mV[NP_GO];
    cfg->pkj_thr_mV = s.thr_mV[NP_PKJ];
    return CB_OK;
  });
}

int cb_net_generate(const cb_net_config *cfg, int n_gr, int n_go, int n_pkj, int comp_gr, int comp_go,
                    int comp_pkj, int64_t cap, int8_t *kind, int32_t *pre, int32_t *post, double *w_nS,
                    int64_t *n) {
  return guarded([&]() -> int {
    if (!cfg || !n) return fail(CB_E_ARG, "null argument");
    NetSpec s = net_spec_of(*cfg);
    const int nn[3] = {n_gr, n_go, n_pkj}, cc[3] = {comp_gr, comp_go, comp_pkj};
    for (int p = 0; p < 3; p++) {
      s.n[p] = nn[p];
      s.comp[p] = cc[p];
    }
    const std::string err = net_check(s);
    if (!err.empty()) return fail(CB_E_ARG, err);
    *n = net_size(s);
    if (!kind && !pre && !post && !w_nS) return CB_OK;
    if (!kind || !pre || !post || !w_nS) return fail(CB_E_ARG, "give every output array or none");
    if (cap < *n) return fail(CB_E_ARG, "cap is smaller than the synapse count");
    NetList L;
    net_generate(s, L);
    for (size_t j = 0; j < L.kind.size(); j++) {
      kind[j] = L.kind[j];
      pre[j] = L.pre[j];
      post[j] = L.post[j];
      w_nS[j] = L.w_nS[j];
    }
    return CB_OK;
  });
}

int cb_net_create(cb_pop *gr, cb_pop *go, cb_pop *pkj, const cb_net_config *cfg, cb_net **out) {
  return guarded([&]() -> int {
    if (!gr || !go || !pkj || !cfg || !out) return fail(CB_E_ARG, "null argument");
    *out = nullptr;
    if (gr->cell_type != CB_GR || go->cell_type != CB_GO || pkj->cell_type != CB_PKJ)
      return fail(CB_E_ARG, "cb_net_create takes a granule, a Golgi and a Purkinje population");
    for (cb_pop *p : {gr, go, pkj}) {
      if (p->in_net) return fail(CB_E_ARG, "a population is coupled to another network");
      if (!p->syn_in.empty()) return fail(CB_E_ARG, "a population already takes synapse sets");
      if (p->device != gr->device) return fail(CB_E_ARG, "the populations must share one device");
    }
    CB_HIP(hipSetDevice(gr->device));
    std::unique_ptr<cb_net> n(new cb_net);
    n->device = gr->device;
    n->net.reset(new Network(gr->eng.get(), go->eng.get(), pkj->eng.get(), net_spec_of(*cfg), gr->device));
    n->pop[0] = gr;
    n->pop[1] = go;
    n->pop[2] = pkj;
    for (cb_pop *p : n->pop) p->in_net = true;
    *out = n.release();
    return CB_OK;
  });
}

int cb_net_run(cb_net *net, int nint) {
  return guarded([&]() -> int {
    if (!net) return fail(CB_E_ARG, "null network");
    if (nint < 0) return fail(CB_E_ARG, "negative interval count");
    CB_HIP(hipSetDevice(net->device));
    net->net->run(nint);
    return CB_OK;
  });
}

int cb_net_spikes(cb_net *net, int cap, double *t_out, int *pop_out, int *cell_out, int *n_out) {
  return guarded([&]() -> int {
    if (!net || !n_out || (cap > 0 && (!t_out || !pop_out || !cell_out))) return fail(CB_E_ARG, "null argument");
    *n_out = net->net->take_spikes(cap, t_out, pop_out, cell_out);
    return CB_OK;
  });
}

int cb_net_conductance(const cb_net *net, int pop, int receptor, double *dst) {
  return guarded([&]() -> int {
    if (!net || !dst) return fail(CB_E_ARG, "null argument");
    net->net->conductance(pop, receptor, dst);
    return CB_OK;
  });
}

int cb_net_stats(const cb_net *net, int64_t *out9) {
  return guarded([&]() -> int {
    if (!net || !out9) return fail(CB_E_ARG, "null argument");
    for (int k = 0; k < NET_NKIND; k++) out9[k] = net->net->count(k);
    for (int p = 0; p < NP_N; p++) out9[4 + p] = net->net->slots(p);
    out9[7] = net->net->intervals();
    out9[8] = net->net->delay_intervals();
    return CB_OK;
  });
}

int cb_net_time(const cb_net *net, double *pop_ms3, double *exchange_ms, double *total_ms) {
  return guarded([&]() -> int {
    if (!net || !pop_ms3 || !exchange_ms || !total_ms) return fail(CB_E_ARG, "null argument");
    net->net->times(pop_ms3, exchange_ms, total_ms);
    return CB_OK;
  });
}

int cb_net_destroy(cb_net *net) {
  return guarded([&]() -> int {
    if (!net) return CB_OK;
    CB_HIP(hipSetDevice(net->device));
    for (cb_pop *p : net->pop)
      if (p) p->in_net = false;
    delete net;
    return CB_OK;
  });
}

int cb_synth_gr_chains(const char *path, const char *template_path, uint64_t seed, int ncell, const int *types,
                       int comp) {
  return guarded([&]() -> int {
    if (!path || !template_path || ncell <= 0) return fail(CB_E_ARG, "bad argument");
    std::vector<int> ty;
    if (types) {
      if (comp <= 0 || comp > gr::COMP) return fail(CB_E_ARG, "bad compartment count");
      ty.assign(types, types + comp);
    } else {
      ty = {3, 4, 6, 7};   // dendrite, soma, axon initial segment, axon (gr.cuh:20-28 types)
    }
    std::string err;
    if (!synth_gr_chains(path, template_path, seed, ncell, ty, err)) return fail(CB_E_IO, err);
    return CB_OK;
  });
}

int cb_synth_go_trees(const char *path, const char *template_path, uint64_t seed, int ncell) {
  return guarded([&]() -> int {
    if (!path || !template_path || ncell <= 0) return fail(CB_E_ARG, "bad argument");
    std::string err;
    if (!synth_go_trees(path, template_path, seed, ncell, err)) return fail(CB_E_IO, err);
    return CB_OK;
  });
}

int cb_synth_io_gj(const char *path, uint64_t seed, int ncell, int k, double g_min_nS, double g_max_nS) {
  return guarded([&]() -> int {
    if (!path || !(g_min_nS >= 0.0) || g_max_nS < g_min_nS) return fail(CB_E_ARG, "bad argument");
    std::string err;
    if (!synth_io_gj(path, seed, ncell, k, g_min_nS, g_max_nS, err)) return fail(CB_E_ARG, err);
    return CB_OK;
  });
}

}  // extern "C"

// Host build of the resident RKC kernel (k_rkc_steps, csrc/rkc_resident.hpp)
// for the CPU tests: one host thread per lane, workgroups of one wavefront, the
// mailboxes in ordinary memory.  The population is a cable matrix with constant
// frozen currents, as the oracle's generic one; the tables below are those the
// engine lays out (GlobalRkc::make_resident).  The controller's scalars and
// counters, one copy per wave on the device, are one per lane here.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>

namespace {

// sense-counting barrier that yields while it waits
struct Barrier {
  int n = 64;
  std::atomic<int> waiting{0};
  std::atomic<long> gen{0};
  void wait() {
    const long g = gen.load(std::memory_order_acquire);
    if (waiting.fetch_add(1, std::memory_order_acq_rel) + 1 == n) {
      waiting.store(0, std::memory_order_relaxed);
      gen.fetch_add(1, std::memory_order_acq_rel);
    } else {
      while (gen.load(std::memory_order_acquire) == g) std::this_thread::yield();
    }
  }
};
struct Group {
  Barrier bar;
  double xs[64];
  int is[64];
  int late = 0;
  std::vector<double> lds;
};
thread_local Group *t_group = nullptr;
thread_local unsigned long long t_polls = 0;
std::atomic<unsigned long long> max_polls{0};

}  // namespace

thread_local emu_dim3 threadIdx;
thread_local emu_dim3 blockIdx;
double emu_shfl_xor(double x, int) { return x; }
void emu_wave_barrier() { t_group->bar.wait(); }
void emu_syncthreads() { t_group->bar.wait(); }
void emu_pause() {   // a poll lets the other lanes run
  t_polls++;
  std::this_thread::yield();
}
int emu_syncthreads_or(int x) {
  t_group->is[threadIdx.x] = x;
  t_group->bar.wait();
  int any = 0;
  for (int i = 0; i < 64; i++) any |= t_group->is[i];
  t_group->bar.wait();
  return any != 0;
}
double emu_shfl_down(double x, int off) {
  t_group->xs[threadIdx.x] = x;
  t_group->bar.wait();
  const double y = (int)threadIdx.x + off < 64 ? t_group->xs[threadIdx.x + off] : x;
  t_group->bar.wait();
  return y;
}
int emu_first_lane(int x) {
  t_group->is[threadIdx.x] = x;
  t_group->bar.wait();
  const int y = t_group->is[0];
  t_group->bar.wait();
  return y;
}
unsigned long long emu_clock() { return t_polls; }   // a lane's time: its looks at mailboxes
static double *emu_lds() { return t_group->lds.data(); }
static int *emu_late() { return &t_group->late; }

#include "rkc_resident.hpp"

namespace cbrkc {
std::vector<double> rkc_stage_table(int mtab);
void rkc_stage_start(int m, double *w1, double *mus);

struct Still {   // constant frozen currents
  struct State {
    const double *b;
  };
  static constexpr int NT = 64, NONFINITE_STATUS = 7;
  static constexpr bool GAP = false, HELP = true, DECAY = false;
  static double ion(const State *S, int i, double, double, const GapView *) { return S->b[i]; }
};
}  // namespace cbrkc
using namespace cbrkc;

extern "C" {
// nsteps macro steps of n cells of comp rows (at most 64 K rows of a cell), cpb
// cells to a workgroup, nhelp helpers to each; present: workgroups that are
// started at all (fewer: the others wait in vain); wait: the limit of a wait, in looks;
// launches: how often the kernel was started; polls: the most looks of a lane.  vec: y, yn, fn, ede, vnew.
// o16, hw8 and cnt5 (steps, rejects, stages, power iterations, ion updates)
// come back.  Returns the last status.
int emu_rkc(int n, int comp, int cpb, int nhelp, int present, const int *row, const int *col, const double *val,
            const double *cm, const double *b, double *vec, double *o16, double *hw8, long long *cnt5, int nsteps,
            double rho_floor, int refresh, long long wait, int *launches,
            long long *polls) {
  const int nc = n * comp, RM = cpb * comp, nblk = (n + cpb - 1) / cpb;
  RkcArgs a{};
  a.n = n;
  a.nc = nc;
  a.comp = comp;
  a.cpb = cpb;
  a.nblk = nblk;
  a.nch = (nc + RED_BLOCK - 1) / RED_BLOCK;
  std::vector<uint2> lcol(nc);
  std::vector<double> lval((size_t)ROW_W * nc, 0.0), xval;
  std::vector<unsigned short> xcol;
  std::vector<int> x0(1, 0), imp0(1, 0), imp;
  for (int w = 0; w < nblk; w++) {
    const int r0 = w * RM, r1 = min(nc, r0 + RM), R = r1 - r0, m0 = (int)imp.size();
    for (int i = r0; i < r1; i++) {
      unsigned c4[4] = {(unsigned)(i - r0), (unsigned)(i - r0), (unsigned)(i - r0), 0u};
      const int xs = (int)xval.size() - x0[w];
      int e = 0;
      for (int j = row[i]; j < row[i + 1]; j++) {
        int l = col[j] - r0;
        if (l < 0 || l >= R) {
          int g = m0;
          while (g < (int)imp.size() && imp[g] != col[j]) g++;
          if (g == (int)imp.size()) imp.push_back(col[j]);
          l = R + g - m0;
        }
        if (e < ROW_W) {
          c4[e] = (unsigned)l;
          lval[(size_t)e * nc + i] = val[j];
        } else {
          xcol.push_back((unsigned short)l);
          xval.push_back(val[j]);
        }
        e++;
      }
      if (e > ROW_W) c4[3] = (unsigned)xs << 4 | (unsigned)(e - ROW_W);
      lcol[i] = make_uint2(c4[0] | c4[1] << 16, c4[2] | c4[3] << 16);
    }
    x0.push_back((int)xval.size());
    imp0.push_back((int)imp.size());
    a.ext_max = max(a.ext_max, x0[w + 1] - x0[w]);
    a.ghost_max = max(a.ghost_max, (int)imp.size() - m0);
  }
  const int nslot = (int)imp.size();
  std::vector<int> exp0(1, 0), er, es;
  for (int w = 0; w < nblk; w++) {
    for (int s = 0; s < nslot; s++)
      if (imp[s] / RM == w) {
        er.push_back(imp[s] % RM);
        es.push_back(s);
      }
    exp0.push_back((int)er.size());
  }
  double empty;
  std::memcpy(&empty, &MAIL_EMPTY, 8);
  std::vector<double> ghost((size_t)3 * GHOST_STAGES * max(1, nslot), empty), terms((size_t)3 * nc, empty),
      parts((size_t)3 * a.nch, empty), gap((size_t)3 * n, empty), req((size_t)9 * nblk, empty),
      vin((size_t)3 * nc, empty), bout((size_t)3 * nc, empty), v1(nc), v2(nc), bb(b, b + nc), iext(nc), amp(n);
  std::vector<double> table = rkc_stage_table(RES_COEF);
  table.resize(RES_COEFS + 2 * (RES_START + 1));
  for (int m = 0; m <= RES_START; m++) rkc_stage_start(m, &table[RES_COEFS + 2 * m], &table[RES_COEFS + 2 * m + 1]);
  if (nslot > 0) {
    a.imp0 = imp0.data();
    a.exp0 = exp0.data();
    a.exp_row = er.data();
    a.exp_slot = es.data();
    a.ghost = ghost.data();
    a.nslot = nslot;
  }
  a.lcol = lcol.data();
  a.lval = lval.data();
  a.xcol = xcol.data();
  a.xval = xval.data();
  a.x0 = x0.data();
  a.terms = terms.data();
  a.parts = parts.data();
  a.gap = gap.data();
  a.nhelp = nhelp;
  a.own = nhelp ? (RM + nhelp) / (nhelp + 1) : RM;
  a.req = req.data();
  a.vin = vin.data();
  a.bout = bout.data();
  a.y = vec;
  a.yn = vec + nc;
  a.fn = vec + 2 * nc;
  a.ede = vec + 3 * nc;
  a.vnew = vec + 4 * nc;
  a.b = bb.data();
  a.v1 = v1.data();
  a.v2 = v2.data();
  a.cm = cm;
  a.coef = table.data();
  a.integ = 1e30;
  a.wait = (unsigned long long)wait;
  max_polls = 0;
  a.rho_floor = rho_floor;
  a.refresh_fn = refresh;
  a.iext = iext.data();
  a.amp = amp.data();
  RkcCtl ctl{}, hosts[2] = {};   // the copy, and the word behind it
  RkcCtl &host = hosts[0];
  const int &late = *(const int *)&hosts[1];
  std::memcpy(ctl.o, o16, sizeof(ctl.o));
  std::memcpy(ctl.hw, hw8, sizeof(ctl.hw));
  ctl.errold3 = std::pow(ctl.o[11], 1.0 / 3.0);
  ctl.last = ctl.newspc = 1;
  ctl.steps = cnt5[0];
  ctl.rejects = cnt5[1];
  ctl.stages = cnt5[2];
  ctl.rho_iters = cnt5[3];
  ctl.ions = cnt5[4];
  host = ctl;
  a.ctl = &ctl;
  a.ctl_host = &host;
  const Still::State S{b};
  const size_t lds = (size_t)5 * (RM + a.ghost_max) + RM + RED_BLOCK + a.nch + 8 + 4 * RES_COEF + a.ext_max +
                     (a.ext_max + 3) / 4;
  const int grid = nblk * (1 + nhelp);
  *launches = 0;
  while (host.macro < nsteps) {
    a.gq0 = host.ions_q;
    std::vector<std::unique_ptr<Group>> groups;
    std::vector<std::thread> th;
    for (int w = 0; w < grid; w++) {
      groups.emplace_back(new Group);
      groups.back()->lds.assign(lds, std::nan(""));
    }
    for (int w = 0; w < min(grid, present); w++)
      for (int lane = 0; lane < 64; lane++)
        th.emplace_back([&, w, lane]() {
          threadIdx = {(unsigned)lane, 0, 0};
          blockIdx = {(unsigned)w, 0, 0};
          t_group = groups[w].get();
          const int left = nsteps - (int)host.macro;
          if (RM <= 64) k_rkc_steps<Still, 1>(a, &S, left, 0.0, 0);
          else k_rkc_steps<Still, 4>(a, &S, left, 0.0, 0);
          unsigned long long most = max_polls;
          while (most < t_polls && !max_polls.compare_exchange_weak(most, t_polls)) {
          }
        });
    for (auto &t : th) t.join();
    *polls = (long long)max_polls.load();
    ++*launches;
    a.resume = host.status == ASK_POW || host.status == ASK_STAGE ? host.status : 0;
    a.p1 = std::pow(host.err, 1.0 / 3.0);
    a.p2 = std::pow(host.err, 2.0 / 3.0);
    if (host.status == ASK_STAGE) rkc_stage_start(host.m, &a.p1, &a.p2);
    if (late) return TIMED_OUT;
    if (host.status != 0 && !a.resume) break;
  }
  std::memcpy(o16, host.o, sizeof(host.o));
  std::memcpy(hw8, host.hw, sizeof(host.hw));
  cnt5[0] = host.steps;
  cnt5[1] = host.rejects;
  cnt5[2] = host.stages;
  cnt5[3] = host.rho_iters;
  cnt5[4] = host.ions;
  return host.status;
}
}

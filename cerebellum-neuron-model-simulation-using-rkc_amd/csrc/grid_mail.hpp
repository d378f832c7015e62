// Values exchanged between the workgroups of one running kernel, and the
// deterministic 256-wide tree sums over rows that several workgroups own.
//
// A mailbox slot is one 8-byte word that holds EMPTY until its value is there,
// so the value is its own flag: the writer stores it with one device-scope
// atomic, the reader polls the word, and no fence (on this chip a write-back
// or an invalidation of an XCD's whole L2) orders anything else.  Every slot
// has one writer and exists three times.  Exchange q uses copy q % 3 of every
// slot; after exchange q a writer empties its slots of copy (q + 2) % 3, last
// used at q - 1, and waits for those stores before it posts anything of
// exchange q + 1.  That is safe because an exchange ends, for any workgroup,
// only when every workgroup has posted its part of it: who has finished
// exchange q knows that all have finished reading q - 1, and who has finished
// exchange q + 1 knows that all of q + 2's slots are empty.  The number of the
// next exchange (modulo 3) is kept with the controller between launches.
//
// Every wait ends: a poll gives up after the population's limit (60 s unless it
// is set), and from then on no wait of that workgroup lasts: whoever gives up
// marks the workgroup's LDS word, every other poll looks at it, and the kernel
// leaves its loops at the next sum and reports TIMED_OUT.  What the limit bounds
// is so a launch, not a poll: the workgroups wait for a lost one side by side, in
// a chain of coupled values and then in the sum, about two limits in all.  All
// workgroups have to be resident, so kernels with more than one are launched
// cooperatively.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "detsum.hpp"

namespace cbrkc {

constexpr int TIMED_OUT = 8;   // status: a workgroup waited for another one in vain
constexpr unsigned long long MAIL_EMPTY = 0x7FF4CE11AB1E0001ull;   // a NaN no arithmetic makes
constexpr unsigned long long WAIT_TICKS = 60ull * 100000000ull;    // the limit of a wait: 60 s of the 100 MHz clock

inline unsigned long long wait_ticks(double seconds) { return (unsigned long long)(seconds * 1e8); }

// The limit of a wait, the workgroup's LDS word that is set once one gave up, and
// whether this thread's did (looked at in every sum: a register)
struct Wait {
  unsigned long long ticks;
  volatile int *late;
  int mine;
};

__device__ inline void mail_put(double *slot, double v) {
  unsigned long long b = (unsigned long long)__double_as_longlong(v);
  if (b == MAIL_EMPTY) b = 0x7FF8000000000000ull;
  __hip_atomic_store((unsigned long long *)slot, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void mail_clear(double *slot) {
  __hip_atomic_store((unsigned long long *)slot, MAIL_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the slot's value once it is there, or 0 when the wait gives up (with a limit
// of 0 at the first look that finds nothing)
__device__ inline double mail_get(const double *slot, Wait &W) {
  // (neither the clock nor the LDS word is looked at before the 128th look, some
  // 100 us: a value is there after a few)
  unsigned long long b, t0 = 0;
  for (unsigned n = 1;; n++) {
    b = __hip_atomic_load((const unsigned long long *)slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (b != MAIL_EMPTY) break;
    if ((n & 127) == 0 || W.ticks == 0) {
      const unsigned long long t = wall_clock64();
      if (t0 == 0) t0 = t;
      if (*W.late || t - t0 >= W.ticks) {
        W.mine = *W.late = 1;
        return 0.0;
      }
    }
  }
  return __longlong_as_double((long long)b);
}
// mail_get for a wait that may be long: it leaves 256 cycles between looks
__device__ inline double mail_wait(const double *slot, Wait &W) {
  const unsigned long long t0 = wall_clock64();
  while (__hip_atomic_load((const unsigned long long *)slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == MAIL_EMPTY) {
    __builtin_amdgcn_s_sleep(4);
    if (*W.late || wall_clock64() - t0 > W.ticks) {
      W.mine = *W.late = 1;
      return 0.0;
    }
  }
  return mail_get(slot, W);
}
// the thread's own stores have reached memory
__device__ inline void mail_settle() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

__device__ inline double first_lane(double x) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(x));
  const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

// block_tree_sum of 256 values by one wave: x0..x3 hold values lane, lane + 64,
// lane + 128, lane + 192; the same additions in the same order, in lane 0
__device__ inline double wave_tree_sum(double x0, double x1, double x2, double x3) {
  double s = (x0 + x2) + (x1 + x3);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s = s + __shfl_down(s, off);
  return s;
}

// One workgroup's share of a sum over nc rows in 256-row chunks.  It owns the
// rows [r0, r1) and computes the chunks that begin among them; the rows before
// its first chunk go to the workgroup that owns their chunk, and the rows its
// last chunk lacks come from the workgroups after it.
struct SumPlan {
  int nc, r0, r1;
  int c0, nown;     // first owned chunk, number of them
  int head, tail;   // rows posted, rows fetched
  int nch;          // chunks of the whole sum
  bool alone;       // one workgroup owns every row
  __device__ void set(int nc_, int r0_, int r1_) {
    nc = nc_; r0 = r0_; r1 = r1_;
    nch = (nc + RED_BLOCK - 1) / RED_BLOCK;
    alone = r0 == 0 && r1 == nc;
    c0 = (r0 + RED_BLOCK - 1) / RED_BLOCK;
    const int ce = (r1 + RED_BLOCK - 1) / RED_BLOCK;   // chunks that begin before r1
    nown = max(0, ce - c0);
    head = min(r1, c0 * RED_BLOCK) - r0;
    tail = nown > 0 ? min(nc, ce * RED_BLOCK) - r1 : 0;
  }
};

// The total of the rows' terms.  term (LDS): the workgroup's own rows, filled
// by the same thread for i = tid, tid + NT, ..., with room for 255 more; part
// (LDS): nch + 8 doubles; terms [3][nc] and parts [3][nch]: mailboxes; q: the
// exchange's number modulo 3, advanced.  late becomes true for the whole
// workgroup when any of its waits gave up.  The order is that of k_reduce256 over the
// whole vector, so the total equals the multi-launch reduction bit for bit.
template <int NT>
__device__ inline double grid_sum(const SumPlan &P, double *term, double *part, double *terms, double *parts,
                                  unsigned &q, Wait &W, bool &late) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, R = P.r1 - P.r0;
  double *tq = terms + (size_t)q * P.nc, *pq = parts + (size_t)q * P.nch;
  if (!P.alone) {
    mail_settle();
    // a workgroup without a chunk posts rows only, each wave its own: all
    // its waves' emptied slots have to be settled before the first of them
    if (P.nown == 0) __syncthreads();
    for (int i = tid; i < P.head; i += NT) mail_put(tq + P.r0 + i, term[i]);
    for (int i = tid; i < P.tail; i += NT) term[R + i] = mail_get(tq + P.r1 + i, W);
  }
  __syncthreads();
  for (int c = wave; c < P.nown; c += NT / 64) {
    const int base = (P.c0 + c) * RED_BLOCK - P.r0 + lane, lim = P.nc - P.r0;
    const double s = wave_tree_sum(base < lim ? term[base] : 0.0, base + 64 < lim ? term[base + 64] : 0.0,
                                   base + 128 < lim ? term[base + 128] : 0.0,
                                   base + 192 < lim ? term[base + 192] : 0.0);
    if (lane == 0) {
      if (P.alone) part[P.c0 + c] = s;
      else mail_put(pq + P.c0 + c, s);
    }
  }
  if (!P.alone)
    for (int k = tid; k < P.nch; k += NT) part[k] = mail_get(pq + k, W);
  if (P.alone) __syncthreads();
  else late = __syncthreads_or(W.mine);
  // the partials by the same tree, level by level (at most 2048 of them)
  int m = P.nch;
  const double *in = part;
  if (m > RED_BLOCK) {
    const int groups = (m + RED_BLOCK - 1) / RED_BLOCK;
    double *out = part + P.nch;
    for (int c = wave; c < groups; c += NT / 64) {
      const int k = c * RED_BLOCK + lane;
      const double s = wave_tree_sum(k < m ? in[k] : 0.0, k + 64 < m ? in[k + 64] : 0.0,
                                     k + 128 < m ? in[k + 128] : 0.0, k + 192 < m ? in[k + 192] : 0.0);
      if (lane == 0) out[c] = s;
    }
    __syncthreads();
    in = out;
    m = groups;
  }
  const double tot = wave_tree_sum(lane < m ? in[lane] : 0.0, lane + 64 < m ? in[lane + 64] : 0.0,
                                   lane + 128 < m ? in[lane + 128] : 0.0, lane + 192 < m ? in[lane + 192] : 0.0);
  if (!P.alone) {
    // empty the copies of the exchange before this one
    const size_t old = q == 0 ? 2 : q - 1;
    for (int i = tid; i < P.head; i += NT) mail_clear(terms + old * P.nc + P.r0 + i);
    for (int c = wave; c < P.nown; c += NT / 64)
      if (lane == 0) mail_clear(parts + old * P.nch + P.c0 + c);
  }
  q = q == 2 ? 0 : q + 1;
  return first_lane(tot);
}

}  // namespace cbrkc

// exp(x) rounded to nearest from a double-double evaluation, for the model
// code whose trajectories amplify last-bit differences (the gap-coupled
// inferior-olive grid).
//
// Method (Cody & Waite argument reduction, then Taylor series with repeated
// squaring, all in double-double arithmetic with FMA error-free products,
// Dekker/Knuth two-sum):
//   k = rint(x / ln 2),  r = x - k ln 2           (ln 2 split into 3 parts)
//   exp(r) = (exp(r / 2^8))^(2^8),  exp(s) = sum_{i <= 10} s^i / i!
//   exp(x) = 2^k exp(r)
// The double-double result carries ~100 bits, so rounding its sum to double
// gives the correctly rounded exp except in cases closer to a rounding
// boundary than ~2^-45 ulp.  Arguments outside (-708, 709) fall back to
// exp(), which is exact at the overflow / underflow ends that matter here.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace cbrkc {

struct dd {
  double hi, lo;
};

__host__ __device__ inline dd dd_two_sum(double a, double b) {
  const double s = a + b;
  const double bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}
__host__ __device__ inline dd dd_fast_two_sum(double a, double b) {
  const double s = a + b;
  return {s, b - (s - a)};
}
__host__ __device__ inline dd dd_add(dd a, dd b) {
  dd s = dd_two_sum(a.hi, b.hi);
  dd t = dd_two_sum(a.lo, b.lo);
  s.lo += t.hi;
  s = dd_fast_two_sum(s.hi, s.lo);
  s.lo += t.lo;
  return dd_fast_two_sum(s.hi, s.lo);
}
__host__ __device__ inline dd dd_mul(dd a, dd b) {
  const double p = a.hi * b.hi;
  double e = fma(a.hi, b.hi, -p);
  e = fma(a.hi, b.lo, e);
  e = fma(a.lo, b.hi, e);
  return dd_fast_two_sum(p, e);
}
__host__ __device__ inline dd dd_mul_d(dd a, double b) {
  const double p = a.hi * b;
  double e = fma(a.hi, b, -p);
  e = fma(a.lo, b, e);
  return dd_fast_two_sum(p, e);
}

__host__ __device__ inline double exp_acc(double x) {
  if (!(x > -708.0 && x < 709.0)) return exp(x);
  // ln 2 = L1 + L2 + L3: L1 is ln 2 rounded to 32 fraction bits, so k L1 is
  // exact for |k| < 2^21 and x - k L1 is exact (Sterbenz); L2, L3 are the next
  // two parts rounded to double
  const double L1 = 0.6931471806019545;
  const double L2 = -4.2009150726810846e-11;
  const double L3 = -1.3124698417785255e-27;
  const double k = rint(x * 1.4426950408889634074);
  const double t = x - k * L1;                 // exact
  // r = t - k L2 - k L3 in double-double
  const double p = k * L2;
  const double pe = fma(k, L2, -p);
  dd r = dd_two_sum(t, -p);
  r.lo -= pe + k * L3;
  r = dd_fast_two_sum(r.hi, r.lo);
  // s = r / 2^8 (exact scaling)
  const dd s = {r.hi * 0.00390625, r.lo * 0.00390625};
  // Taylor sum for exp(s) - 1 in Horner form, |s| < 0.0014: 10 terms reach 2^-110
  dd acc = {2.755731922398589e-07, 0.0};   // 1/10!
  // 1/i! for i = 9..0 as double-double: the double nearest and the exact
  // remainder 1/i! - double(1/i!) rounded to double
  const double inv[10] = {2.7557319223985893e-06, 2.48015873015873e-05, 0.0001984126984126984,
                          0.001388888888888889,   0.008333333333333333, 0.041666666666666664,
                          0.16666666666666666,    0.5,                  1.0,
                          1.0};
  const double inv_lo[10] = {-1.858393274046472e-22, 2.1511947866775882e-23, 1.7209558293420705e-22,
                             -5.300543954373577e-20, 1.1564823173178714e-19, 2.3129646346357427e-18,
                             9.25185853854297e-18,   0.0,                    0.0,
                             0.0};
  for (int i = 0; i < 10; i++) {
    acc = dd_mul(acc, s);
    acc = dd_add(acc, dd{inv[i], inv_lo[i]});
  }
  // square 8 times: exp(r) = exp(s)^256
  for (int i = 0; i < 8; i++) acc = dd_mul(acc, acc);
  return ldexp(acc.hi + acc.lo, (int)k);
}

// The same correctly rounded exp in a sixth of the operations, by Ziv's
// method: a result accurate enough to round nearly always, its error bound
// tested against the rounding, and exp_acc for what the test leaves open.
//   exp(r) = (exp(s))^32, s = r / 32, |s| < 0.0109
//   exp(s) = 1 + s + s^2/2 in double-double + s^3 (1/6 + ... + s^6/9!) in double
// The double part's rounding is 2^-53 of s^3/6 < 2^-22, the series stops
// below 2^-77, and five squarings multiply the relative error by 32: below
// 2^-68 in all, against the 2^-67 tested, which leaves one argument in 8000
// to exp_acc.  Both return the double nearest to exp(x), so the results are
// the same bit for bit.
// Measured, one update of 33536 Golgi compartments (39 distinct exponentials):
// 69 us with exp_acc at every place, 31 with exp_cr inlined there, 25 with one
// copy of it (exp_call below).
// exp(x) = (h + l) 2^k for x in (-708, 709), to 2^-68
__host__ __device__ inline void exp_parts(double x, double &h, double &l, double &k) {
  const double L1 = 0.6931471806019545, L2 = -4.2009150726810846e-11, L3 = -1.3124698417785255e-27;
  k = rint(x * 1.4426950408889634074);
  const double t = x - k * L1;   // exact
  const double p = k * L2;
  const double pe = fma(k, L2, -p);
  const dd u = dd_two_sum(t, -p);
  const double rl = u.lo - (pe + k * L3);
  const double sh = u.hi * 0.03125, sl = rl * 0.03125;
  double q = fma(sh, 2.7557319223985893e-06, 2.48015873015873e-05);
  q = fma(sh, q, 0.0001984126984126984);
  q = fma(sh, q, 0.001388888888888889);
  q = fma(sh, q, 0.008333333333333333);
  q = fma(sh, q, 0.041666666666666664);
  q = fma(sh, q, 0.16666666666666666);
  const double a = sh * sh, ae = fma(sh, sh, -a);
  q *= a * sh;
  const double b = 0.5 * a;
  const double h0 = 1.0 + sh, e0 = sh - (h0 - 1.0);
  const double h1 = h0 + b, e1 = b - (h1 - h0);
  h = h1 + q;
  l = e0 + (e1 + ((q - (h - h1)) + fma(sl, sh + b, 0.5 * ae + sl)));
#pragma unroll
  for (int i = 0; i < 5; i++) {
    const double z = h * h;
    l = fma(h + h, l, fma(h, h, -z));
    h = z;
  }
}
__host__ __device__ inline double exp_cr(double x) {
  if (!(x > -708.0 && x < 709.0)) return exp(x);
  double h, l, k;
  exp_parts(x, h, l, k);
  const double d = h * 6.7762635780344027e-21;   // 2^-67
  const double up = h + (l + d), dn = h + (l - d);
  if (up != dn) return exp_acc(x);
  return ldexp(up, (int)k);
}

// s = h + l rounded, and whether it lies so far (slack, in its last place) from a
// middle between two doubles that a function with an error below 0.5 + slack
// rounds to s as well; s within (1e-20, 1e20)
__host__ __device__ inline double round_sure(double h, double l, double slack, bool &sure) {
  const double s = h + l, rem = (h - s) + l;
  long long e;
  __builtin_memcpy(&e, &s, 8);
  e = (e & 0x7FF0000000000000ll) - (52ll << 52);
  double ulp;
  __builtin_memcpy(&ulp, &e, 8);
  sure = fabs(fabs(rem) - 0.5 * ulp) > slack * ulp;
  return s;
}

// The host libm's exp(x) where sure (all but one argument in 40).  glibc's error is
// below 0.511 of the last place, so it misses the nearest double only where the value lies
// within 0.011 of the middle between two (0.0071 measured, 20 million arguments of
// decays and up to -5)
__host__ __device__ inline double exp_libm(double x, bool &sure) {
  sure = false;
  if (!(x > -708.0 && x < 709.0)) return 0.0;
  double h, l, k;
  exp_parts(x, h, l, k);
  return ldexp(round_sure(h, l, 0.012, sure), (int)k);
}

// The models' exponential (inferior olive, Golgi cells): the host C
// library's on the host (initial state), the correctly rounded exp_cr on the
// device.  These populations amplify last-bit differences of exp into
// spike-time shifts over hundreds of milliseconds, so the device follows a
// correctly rounded exp rather than the device library's (faithful, not
// correctly rounded) one.
// CB_HOST_EMU_DEVICE / CB_HOST_EMU_HOST: the host build of the device code
// used by the tests (a host stand-in for the HIP header, one thread per
// lane) takes the device's or the host's exponential explicitly.
#if defined(CB_HOST_EMU_DEVICE)
static inline double mexp(double x) { return exp_cr(x); }
#elif defined(CB_HOST_EMU_HOST)
static inline double mexp(double x) { return ::exp(x); }
#else
__host__ inline double mexp(double x) { return ::exp(x); }
// One function rather than sixty-odd copies: a model's update is then a few
// thousand instructions and fits the instruction cache, and equal arguments (a
// gate's rates enter its steady state and its time constant) are evaluated
// once.
__device__ __attribute__((noinline, const)) static double exp_call(double x) { return exp_cr(x); }
__device__ inline double mexp(double x) { return exp_call(x); }
#endif

}  // namespace cbrkc

// Host stand-in for the HIP runtime header, for the host build of the
// small-cell device body (tests/host_emu): just enough for that code to
// compile as host C++ with one host thread per lane.  Shuffles and wave
// barriers synchronise the lanes of one cell group (emu_main.cpp).
#pragma once
#include <math.h>

#include <cmath>
#include <cstddef>
#include <cstdint>
#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__
#define __launch_bounds__(...)
struct emu_dim3 {
  unsigned x, y, z;
};
extern thread_local emu_dim3 threadIdx;
extern thread_local emu_dim3 blockIdx;
double emu_shfl_xor(double x, int off);
void emu_wave_barrier();
inline double __shfl_xor(double x, int off) { return emu_shfl_xor(x, off); }
#define __builtin_amdgcn_wave_barrier() emu_wave_barrier()
inline unsigned atomicOr(unsigned *p, unsigned v) { return __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST); }
inline int atomicAdd(int *p, int v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
typedef int hipError_t;
typedef void *hipStream_t;
constexpr hipError_t hipSuccess = 0;
inline const char *hipGetErrorString(hipError_t) { return "host stand-in"; }

// For the resident RKC kernel (resident_emu.cpp): workgroups of host threads,
// the wavefront exchanges of a 64-lane workgroup, and the device's atomics.
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
#define __hip_atomic_load(p, order, scope) (emu_pause(), __atomic_load_n(p, order))
void emu_pause();
void emu_syncthreads();
int emu_syncthreads_or(int x);
double emu_shfl_down(double x, int off);
int emu_first_lane(int x);
unsigned long long emu_clock();
#define __syncthreads() emu_syncthreads()
#define __syncthreads_or(x) emu_syncthreads_or(x)
inline double __shfl_down(double x, int off) { return emu_shfl_down(x, off); }
#define __builtin_amdgcn_readfirstlane(x) emu_first_lane(x)
#define __builtin_amdgcn_s_sleep(x) ((void)0)
#define __builtin_amdgcn_logf(x) log2f(x)
#define __builtin_amdgcn_exp2f(x) exp2f(x)
#define wall_clock64() emu_clock()
inline long long __double_as_longlong(double x) { long long b; __builtin_memcpy(&b, &x, 8); return b; }
inline double __longlong_as_double(long long b) { double x; __builtin_memcpy(&x, &b, 8); return x; }
inline int __double2loint(double x) { return (int)__double_as_longlong(x); }
inline int __double2hiint(double x) { return (int)(__double_as_longlong(x) >> 32); }
inline double __hiloint2double(int hi, int lo) { return __longlong_as_double((long long)hi << 32 | (unsigned)lo); }
struct uint2 {
  unsigned x, y;
};
struct double2 {
  double x, y;
};
inline uint2 make_uint2(unsigned x, unsigned y) { return {x, y}; }
inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }

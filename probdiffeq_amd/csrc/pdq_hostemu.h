// Host build of the device sources (test infrastructure): compiled with g++
// and PDQ_HOST_EMU defined, the kernels' per-instance code runs on the CPU
// with one lane per group (G = 1) and one thread per workgroup, or a whole
// workgroup as one thread per lane with the harness's barriers (tests/emu), so
// that the kernel logic can be checked against the oracle without a GPU.
// LDS arrays are static: shared by the threads of the one workgroup that runs.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static

struct PdqEmuDim {
  unsigned x = 0;
};
inline thread_local PdqEmuDim threadIdx, blockIdx;
inline PdqEmuDim blockDim{1}, gridDim{1};

// The barriers of a workgroup's lanes and of one wavefront's (nothing outside a group).
void pdq_emu_group_barrier();
void pdq_emu_wave_barrier();

inline void __syncthreads() { pdq_emu_group_barrier(); }
inline void __threadfence_block() {}
inline double __shfl_xor(double v, int, int) { return v; }
inline int __shfl(int v, int, int) { return v; }
inline double __shfl(double v, int, int) { return v; }
inline int pdq_emu_atomics = 0;  // atomic operations issued, by all lanes
inline int atomicAdd(int* p, int v) {
  __atomic_fetch_add(&pdq_emu_atomics, 1, __ATOMIC_RELAXED);
  return __atomic_fetch_add(p, v, __ATOMIC_RELAXED);
}
template <class T>
inline void pdq_emu_store(T v, T* p) {
  *p = v;
}
#define __builtin_nontemporal_store pdq_emu_store
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_fence(a, b) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)

using std::copysign;
using std::fabs;
using std::fmax;
using std::fmin;
using std::hypot;
using std::isfinite;
using std::log;
using std::pow;
using std::sqrt;
typedef void* hipStream_t;

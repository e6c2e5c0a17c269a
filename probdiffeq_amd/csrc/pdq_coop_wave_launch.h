// Kernel and launcher of one fixed shape of the cooperative solver
// (pdq_coop_wave.h).  The shapes are compiled in three translation units
// (filter, smoothers, exponential prior), so that they build in parallel.
#pragma once

#include <algorithm>

#include "pdq_coop_wave.h"

namespace pdq {

template <class SH>
__global__ void __launch_bounds__(64) solve_wave_kernel(KArgs args) {  // read in place (WArgs)
  extern __shared__ double pdq_wave_lds[];
  WCtx<SH> c((WArgs*)__builtin_amdgcn_kernarg_segment_ptr(), pdq_wave_lds, threadIdx.x);
  const WArgs& a = *c.a;
  w_setup<SH>(a, pdq_wave_lds, c.l);
  for (;;) {
    // Every lane takes part in the pull (lane 0 adds one, the others nothing).
    // Under a branch for lane 0 alone, the other lanes' index is a constant of
    // the loop, and the compiler may split the loop by lane: lane 0 leaves for
    // the next pull while the others go round with their constant, for ever.
    c.inst = __builtin_amdgcn_readfirstlane(atomicAdd(a.queue, c.l == 0 ? 1 : 0));
    if (c.inst >= a.n_inst) break;
    w_solve_instance(c);
  }
}

template <class SH>
int launch_wave(KArgs& a, hipStream_t st) {
  const size_t lds = sizeof(double) * (size_t)(SH::fixed_size + a.cfg.n_params);
  auto kern = solve_wave_kernel<SH>;
  PDQ_HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  int per_cu = 0;
  PDQ_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 64, lds));
  if (per_cu < 1) return host_error(PDQ_ERR_UNSUPPORTED, "instance does not fit into LDS (%zu bytes)", lds);
  const int grid = (int)std::max<long>(1, std::min<long>(a.n_inst, (long)per_cu * num_cus()));
  launch_zero_queue(a.queue, st);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64), lds, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  return PDQ_OK;
}

// The exponential prior: the filter.
inline int launch_coop_wave_expo(KArgs& a, hipStream_t st) {
  switch (a.lay.N) {
    case 3: return launch_wave<WShape<3, 2, true, false, true>>(a, st);
    case 4: return launch_wave<WShape<4, 2, true, false, true>>(a, st);
    case 5: return launch_wave<WShape<5, 2, true, false, true>>(a, st);
    case 6: return launch_wave<WShape<6, 2, true, false, true>>(a, st);
  }
  return host_error(PDQ_ERR_UNSUPPORTED, "no fixed-shape kernel for num_derivatives = %d", a.lay.N - 1);
}

template <bool SMOOTHER>
int launch_coop_wave_s(KArgs& a, hipStream_t st) {
  if (a.cfg.factorisation == PDQ_ISOTROPIC)
    return a.lay.N == 3 ? launch_wave<WShape<3, 2, false, SMOOTHER>>(a, st)
                        : launch_wave<WShape<6, 2, false, SMOOTHER>>(a, st);
  switch (a.lay.N) {
    case 3: return launch_wave<WShape<3, 2, true, SMOOTHER>>(a, st);
    case 4: return launch_wave<WShape<4, 2, true, SMOOTHER>>(a, st);
    case 5: return launch_wave<WShape<5, 2, true, SMOOTHER>>(a, st);
    case 6: return launch_wave<WShape<6, 2, true, SMOOTHER>>(a, st);
  }
  return host_error(PDQ_ERR_UNSUPPORTED, "no fixed-shape kernel for num_derivatives = %d", a.lay.N - 1);
}

}  // namespace pdq

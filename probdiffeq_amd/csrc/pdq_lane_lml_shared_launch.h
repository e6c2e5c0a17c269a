// Launcher of the LML with the batch's factors computed once, for one nu
// (pdq_lane_lml_shared_nu<nu>.hip, so that the units build in parallel).
#pragma once

#include "pdq_lane_lml_shared.h"

namespace pdq {

template <int N>
int launch_lml_shared_n(LmlArgs& a, int tpl, bool reverse, hipStream_t st);

#ifdef PDQ_LML_SHARED_DEFINE_LAUNCH
template <int N>
int launch_lml_factors(LmlArgs& a, hipStream_t st) {
  const int steps = a.K - 1, intervals = steps / a.every;
  hipLaunchKernelGGL(lml_chain_kernel<N>, dim3(1), dim3(64), 0, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(lml_revert_kernel<N>, dim3((steps + 63) / 64), dim3(64), 0, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(lml_merge_kernel<N>, dim3((intervals + 63) / 64), dim3(64), 0, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  return PDQ_OK;
}

template <int N, int FIELD>
int launch_lml_lanes(LmlArgs& a, int tpl, bool reverse, hipStream_t st) {
  const dim3 grid((unsigned)(((long)a.n_inst * a.G + 63) / 64));
  if (reverse) hipLaunchKernelGGL((lml_adjoint_kernel<N, 2, FIELD>), grid, dim3(64), 0, st, a);
  else if (tpl == 0) hipLaunchKernelGGL((lml_means_kernel<N, 2, 0, FIELD>), grid, dim3(64), 0, st, a);
  else if (tpl == 1) hipLaunchKernelGGL((lml_means_kernel<N, 2, 1, FIELD>), grid, dim3(64), 0, st, a);
  else return host_error(PDQ_ERR_UNSUPPORTED, "no lane LML kernel with %d tangents per lane", tpl);
  PDQ_HIP_TRY(hipGetLastError());
  return PDQ_OK;
}

template <int N>
int launch_lml_shared_n(LmlArgs& a, int tpl, bool reverse, hipStream_t st) {
  if (((long)a.n_inst * a.G + 63) / 64 > 0x7fffffffL) return host_error(PDQ_ERR_UNSUPPORTED, "too many instances");
  const int rc = launch_lml_factors<N>(a, st);
  if (rc) return rc;
  switch (a.cfg.vector_field) {
    case PDQ_VF_LOTKA_VOLTERRA: return launch_lml_lanes<N, PDQ_VF_LOTKA_VOLTERRA>(a, tpl, reverse, st);
    case PDQ_VF_VAN_DER_POL: return launch_lml_lanes<N, PDQ_VF_VAN_DER_POL>(a, tpl, reverse, st);
    case PDQ_VF_BURGERS: return launch_lml_lanes<N, PDQ_VF_BURGERS>(a, tpl, reverse, st);
    case PDQ_VF_LINEAR: return launch_lml_lanes<N, PDQ_VF_LINEAR>(a, tpl, reverse, st);
    case PDQ_VF_LOGISTIC: return launch_lml_lanes<N, PDQ_VF_LOGISTIC>(a, tpl, reverse, st);
  }
  return host_error(PDQ_ERR_INVALID, "unknown vector field %d", a.cfg.vector_field);
}
#endif

}  // namespace pdq

// Launcher of the LML with the batch's factors computed once, for one nu
// (pdq_lane_lml_shared_nu<nu>.hip, so that the units build in parallel).
#pragma once

#include "pdq_lane_lml_shared.h"

namespace pdq {

template <int N>
int launch_lml_shared_n(LmlArgs& a, int tpl, bool reverse, hipStream_t st);

#ifdef PDQ_LML_SHARED_DEFINE_LAUNCH
// The factors and the means' pass (lml_for_launches).
template <int N, int TPL, int FIELD, bool ADJOINT>
int launch_lml_parts(const LmlArgs& a, hipStream_t st) {
  const int lanes = (int)(((long)a.n_inst * a.G + 63) / 64);
  auto factors = [&] {
    hipLaunchKernelGGL((lml_factors_kernel<N>), dim3(1), dim3(64), 0, st, a);
    PDQ_HIP_TRY(hipGetLastError());
    return (int)PDQ_OK;
  };
  return lml_for_launches(a.K - 1, a.every, lanes, factors, [&](const LmlParts& w, int grid) {
    hipLaunchKernelGGL((lml_parts_kernel<N, 2, TPL, FIELD, ADJOINT>), dim3(grid), dim3(64), 0, st, a, w);
    PDQ_HIP_TRY(hipGetLastError());
    return (int)PDQ_OK;
  });
}

template <int N, int FIELD>
int launch_lml_lanes(LmlArgs& a, int tpl, bool reverse, hipStream_t st) {
  if (!reverse) {
    if (tpl == 0) return launch_lml_parts<N, 0, FIELD, false>(a, st);
    if (tpl == 1) return launch_lml_parts<N, 1, FIELD, false>(a, st);
    return host_error(PDQ_ERR_UNSUPPORTED, "no lane LML kernel with %d tangents per lane", tpl);
  }
  const int rc = launch_lml_parts<N, 0, FIELD, true>(a, st);
  if (rc) return rc;
  hipLaunchKernelGGL((lml_adjoint_kernel<N, 2, FIELD>), dim3((a.n_inst + 63) / 64), dim3(128), 0, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  return PDQ_OK;
}

template <int N>
int launch_lml_shared_n(LmlArgs& a, int tpl, bool reverse, hipStream_t st) {
  // (the grid also holds the factors' blocks)
  if (((long)a.n_inst * a.G + 63) / 64 > 0x3fffffffL) return host_error(PDQ_ERR_UNSUPPORTED, "too many instances");
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

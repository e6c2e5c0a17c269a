// Launcher of the LML with the batch's factors computed once, for one nu
// (pdq_lane_lml_shared_nu<nu>.hip, so that the units build in parallel).
#pragma once

#include <algorithm>

#include "pdq_lane_lml_shared.h"

namespace pdq {

template <int N>
int launch_lml_shared_n(LmlArgs& a, int tpl, bool reverse, hipStream_t st);

#ifdef PDQ_LML_SHARED_DEFINE_LAUNCH
// The factors and the means' pass.  Up to 64 steps: the factors in one launch
// (a step, or an interval, per lane of one wavefront), the means in a second:
// what such a call costs is its launches.  Beyond, in chunks of whole intervals: launch i runs
// the chain of chunk i, the reverts of the one before, its predecessor's merges
// and the means of the one before that.  The first three launches run without
// means (24 chunks: an eighth of the chain's time); a chunk of fewer than 64
// steps (70 us) would not cover its launch, and with fewer than six the three
// launches that fill and drain take what the overlap gives (nu = 4, 200 steps,
// gradient: 0.83 ms in four chunks, 0.77 in one).
template <int N, int TPL, int FIELD, bool ADJOINT>
int launch_lml_parts(const LmlArgs& a, hipStream_t st) {
  const int steps = a.K - 1, target = std::max((steps + 23) / 24, 64);
  int chunk = (int)std::min<long>(steps, ((long)target + a.every - 1) / a.every * a.every);
  if ((steps + chunk - 1) / chunk < 6) chunk = steps;
  const int n = (steps + chunk - 1) / chunk, lanes = (int)(((long)a.n_inst * a.G + 63) / 64);
  auto from = [&](int i) { return i < 0 || i >= n ? 0 : i * chunk; };
  auto to = [&](int i) { return i < 0 || i >= n ? 0 : std::min(steps, (i + 1) * chunk); };
  auto launch = [&](const LmlParts& w, int grid) {
    hipLaunchKernelGGL((lml_parts_kernel<N, 2, TPL, FIELD, ADJOINT>), dim3(grid), dim3(64), 0, st, a, w);
    PDQ_HIP_TRY(hipGetLastError());
    return (int)PDQ_OK;
  };
  if (steps <= 64) {
    const int rc = launch(LmlParts{0, steps, 0, steps, 0, steps / a.every, 0, 0, 1}, 1);
    return rc ? rc : launch(LmlParts{0, 0, 0, 0, 0, 0, 0, steps, 0}, 1 + lanes);
  }
  for (int i = 0; i < n + 3; ++i) {
    const LmlParts w{from(i),     to(i),     from(i - 1), to(i - 1), from(i - 2) / a.every, to(i - 2) / a.every,
                     from(i - 3), to(i - 3), 0};
    const int rc = launch(w, 1 + w.reverts() + w.merges() + (w.m0 < w.m1 ? lanes : 0));
    if (rc) return rc;
  }
  return PDQ_OK;
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

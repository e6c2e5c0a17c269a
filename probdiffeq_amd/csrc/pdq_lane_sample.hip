// Instantiations and launcher of the posterior sampler.
#include <algorithm>

#include "pdq_lane_sample.h"

namespace pdq {

namespace {

template <int N, int D>
int launch_sample_nd(SampleArgs& a, hipStream_t st) {
  const long total = (long)a.n_inst * a.n_samples;
  const long need = (total + 63) / 64;
  const long cap = 64L * num_cus();
  const int grid = (int)std::max<long>(1, std::min(need, cap));
  // Reading conditionals together pays when memory, not the step's latency, is
  // the bound: 16 samples of nu = 4 on 200 points take 0.247 / 0.191 ms (staged /
  // each lane its own) in 16 wavefronts, 0.254 / 0.243 in one per CU, 0.287 /
  // 0.357 in two and 0.506 / 0.643 in four.
  if (a.n_samples >= kSampleStagedMin && need >= 2L * num_cus())
    hipLaunchKernelGGL((lane_sample_kernel<N, D, true>), dim3(grid), dim3(64), 0, st, a);
  else
    hipLaunchKernelGGL((lane_sample_kernel<N, D, false>), dim3(grid), dim3(64), 0, st, a);
  PDQ_HIP_TRY(hipGetLastError());
  return PDQ_OK;
}

}  // namespace

int launch_sample(SampleArgs& a, int N, int D, hipStream_t st) {
  if (D == 2) {
    if (N == 4) return launch_sample_nd<4, 2>(a, st);
    if (N == 5) return launch_sample_nd<5, 2>(a, st);
  }
  return host_error(PDQ_ERR_UNSUPPORTED, "no sampler for nu + 1 = %d, d = %d", N, D);
}

}  // namespace pdq

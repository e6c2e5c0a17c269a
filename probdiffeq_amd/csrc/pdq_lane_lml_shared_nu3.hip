// The LML with the batch's factors computed once, nu = 3, and the dispatch.
#define PDQ_LML_SHARED_DEFINE_LAUNCH
#include "pdq_lane_lml_shared_launch.h"

namespace pdq {

template int launch_lml_shared_n<4>(LmlArgs&, int, bool, hipStream_t);

// Four launches against one: below 8 grid steps the value and the forward
// gradient of the lane kernels are as fast or faster (nu = 3, gradient of 1..5
// instances: 2 steps 79 us against 99, 6 steps 94 / 95, 16 steps 132 / 128, 34
// steps 280 / 200); the adjoint's never is (2 steps: 122 / 97).
bool lml_shared_takes(const pdq_config& c, int N, int D, int K, bool reverse) {
  return D == 2 && (N == 4 || N == 5) && c.solver == PDQ_SOLVER && (reverse || K > 8);
}

size_t lml_shared_doubles(int N, int K, int every) {
  return N == 4 ? LmlShared<4>(K, every).size : LmlShared<5>(K, every).size;
}

size_t lml_shared_scratch(int N, int D, int tpl, int K, int every, int n_inst, int G, bool reverse) {
  if (reverse) {
    const size_t lanes = (size_t)((n_inst + 63) / 64) * 64;
    return (N == 4 ? LmlAdjShared<4, 2>(K, every).size : LmlAdjShared<5, 2>(K, every).size) * lanes;
  }
  // an interval's noise mean per interval; m and r between two launches
  return ((size_t)((K - 1) / every) + 2) * N * D * (1 + tpl) * n_inst * G;
}

int launch_lml_shared(LmlArgs& a, int N, int D, int tpl, bool reverse, hipStream_t st) {
  if (D != 2) return host_error(PDQ_ERR_UNSUPPORTED, "no lane LML kernel for nu + 1 = %d, d = %d", N, D);
  return N == 4 ? launch_lml_shared_n<4>(a, tpl, reverse, st) : launch_lml_shared_n<5>(a, tpl, reverse, st);
}

}  // namespace pdq

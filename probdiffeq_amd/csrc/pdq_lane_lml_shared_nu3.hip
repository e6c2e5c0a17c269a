// The LML with the batch's factors computed once, nu = 3, and the dispatch.
#define PDQ_LML_SHARED_DEFINE_LAUNCH
#include "pdq_lane_lml_shared_launch.h"

namespace pdq {

template int launch_lml_shared_n<4>(LmlArgs&, int, bool, hipStream_t);

// PDQ_SOLVER takes this form at every size.  Us of a call, the lane kernels that
// compute every lane's own factors / this form (the factors of up to 64 steps in
// one launch, the call's buffers in one allocation): nu = 3, value, 1 step 55 / 49
// (1 instance), 64 / 50 (1024), 8 steps 68 / 56, 64 steps 261 / 183; gradient by
// tangents, 1 step 64 / 55, 8 steps of 8192 instances 164 / 76; nu = 4, 8 steps
// 131 / 95; the adjoint, nu = 3, 1 step 66 / 58, 4 steps 94 / 67, nu = 4, 1 step
// 81 / 61.
bool lml_shared_takes(const pdq_config& c, int N, int D) {
  return D == 2 && (N == 4 || N == 5) && c.solver == PDQ_SOLVER;
}

size_t lml_shared_doubles(int N, int K, int every) { return lml_shared_size(N, K, every); }

size_t lml_shared_scratch(int N, int D, int tpl, int K, int every, int n_inst, int G, bool reverse) {
  return lml_shared_scratch_size(N, D, tpl, K, every, n_inst, G, reverse);
}

int launch_lml_shared(LmlArgs& a, int N, int D, int tpl, bool reverse, hipStream_t st) {
  if (D != 2) return host_error(PDQ_ERR_UNSUPPORTED, "no lane LML kernel for nu + 1 = %d, d = %d", N, D);
  return N == 4 ? launch_lml_shared_n<4>(a, tpl, reverse, st) : launch_lml_shared_n<5>(a, tpl, reverse, st);
}

}  // namespace pdq

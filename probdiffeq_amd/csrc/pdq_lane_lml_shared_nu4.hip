// The LML with the batch's factors computed once, nu = 4.
#define PDQ_LML_SHARED_DEFINE_LAUNCH
#include "pdq_lane_lml_shared_launch.h"

namespace pdq {

template int launch_lml_shared_n<5>(LmlArgs&, int, bool, hipStream_t);

}  // namespace pdq

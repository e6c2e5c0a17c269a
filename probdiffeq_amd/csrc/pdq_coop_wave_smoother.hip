// Fixed-shape cooperative solves: the smoothers.
#include "pdq_coop_wave_launch.h"

namespace pdq {
int launch_coop_wave_smoother(KArgs& a, hipStream_t st) { return launch_coop_wave_s<true>(a, st); }
}  // namespace pdq

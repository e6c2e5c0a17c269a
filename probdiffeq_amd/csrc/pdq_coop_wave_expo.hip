// Fixed-shape cooperative solves: the filter with an exponential prior.
#include "pdq_coop_wave_launch.h"

namespace pdq {
int launch_coop_wave_exponential(KArgs& a, hipStream_t st) { return launch_coop_wave_expo(a, st); }
}  // namespace pdq

// Fixed-shape cooperative solves: the filter.
#include "pdq_coop_wave_launch.h"

namespace pdq {
int launch_coop_wave_filter(KArgs& a, hipStream_t st) { return launch_coop_wave_s<false>(a, st); }
}  // namespace pdq

// Block-diagonal kernel instantiations for strategy_filter (nu = 1..5),
// the option defaults folded in.
#define PDQ_BD_DEFINE_LAUNCH
#include "pdq_bd_launch.h"

namespace pdq {
PDQ_BD_INSTANTIATE(PDQ_FILTER, false)
}  // namespace pdq

// Constants of the exponential prior's transition.
#pragma once

#include "pdq_device.h"

namespace pdq {

// pade_and_legendre_9 (util/gram_util.py:261-331): Pade coefficients and the
// Legendre coefficient matrix.
__device__ __forceinline__ double pade9(int i) {
  constexpr double c[10] = {17643225600.0, 8821612800.0, 2075673600.0, 302702400.0, 30270240.0,
                            2162160.0,     110880.0,     3960.0,       90.0,        1.0};
  return c[i];
}
__device__ __forceinline__ double legendre9(int i, int j) {
  constexpr double c[10][10] = {{17643225600.0, 0, 605404800.0, 0, 4324320.0, 0, 7920.0, 0, 2.0, 0},
                                {0, 8821612800.0, 0, 155675520.0, 0, 617760.0, 0, 528.0, 0, 0},
                                {0, 0, 1470268800.0, 0, 15444000.0, 0, 34320.0, 0, 10.0, 0},
                                {0, 0, 0, 147026880.0, 0, 960960.0, 0, 1092.0, 0, 0},
                                {0, 0, 0, 0, 10501920.0, 0, 42120.0, 0, 18.0, 0},
                                {0, 0, 0, 0, 0, 583440.0, 0, 1320.0, 0, 0},
                                {0, 0, 0, 0, 0, 0, 26520.0, 0, 26.0, 0},
                                {0, 0, 0, 0, 0, 0, 0, 1020.0, 0, 0},
                                {0, 0, 0, 0, 0, 0, 0, 0, 34.0, 0},
                                {0, 0, 0, 0, 0, 0, 0, 0, 0, 1.0}};
  return c[i][j];
}

}  // namespace pdq

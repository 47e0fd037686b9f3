// Host stand-ins that let the device headers of acts_amd/csrc compile with
// g++, one lane at a time, for tests without a device.
#pragma once

#include <cmath>

#include "hip_runtime_api.h"

#define __host__
#define __device__

using std::fma;
using std::fmax;
using std::fmin;
using std::signbit;

inline float rsqrtf(float x) { return 1.0f / std::sqrt(x); }

// v_div_fixup: the quotient, with the results of the special operands
inline double __builtin_amdgcn_div_fixup(double q, double b, double a) {
  const bool special = b == 0 || a == 0 || std::isinf(a) || std::isinf(b) || a != a || b != b;
  return special ? a / b : q;
}

// cpfft_common.h -- shared definitions for the MI355X kernels and their
// host-side unit-test build.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define CPFFT_HD __host__ __device__
#else
#include <cmath>
#define CPFFT_HD
using std::atan2;
using std::copysign;
using std::cos;
using std::fabs;
using std::fmax;
using std::pow;
using std::sin;
using std::sqrt;
#endif

#include <stdint.h>

namespace cpfft {

struct cplx {
  double re, im;
};

}  // namespace cpfft

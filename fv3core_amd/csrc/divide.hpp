// Several quotients by one divisor for one reciprocal.
#pragma once

#include <hip/hip_runtime.h>

namespace fv3 {

// Quotients by a divisor that several share: the division's own steps
// (reciprocal, Newton, the residual correction of Markstein, fix-up of zeros,
// infinities and NaN), so the bits are those of a / b but where b or a quotient
// is near the ends of the exponent range.  FP32 divides as it is.  The fix-up
// costs the Riemann chains, two quotients a level, 1 to 2 % of their launches
// (six C96 tiles, 79 levels: 254 -> 258 us and 240 -> 242 us); without it a
// divisor that overflows gives NaN where a / b is 0.
template <typename T>
struct Divisor {
  T b;
  __device__ __forceinline__ explicit Divisor(T v) : b(v) {}
  __device__ __forceinline__ T quot(T a) const { return a / b; }
};
template <>
struct Divisor<double> {
  double b, y;
  __device__ __forceinline__ explicit Divisor(double v) : b(v) {
    y = __builtin_amdgcn_rcp(v);
    y = fma(y, fma(-v, y, 1.0), y);
    y = fma(y, fma(-v, y, 1.0), y);
  }
  __device__ __forceinline__ double quot(double a) const {
    const double q = a * y;
    return __builtin_amdgcn_div_fixup(fma(fma(-b, q, a), y, q), b, a);
  }
};

}  // namespace fv3

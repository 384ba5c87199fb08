// sqrt from an estimate of its reciprocal, for host and device.
#pragma once

#ifdef __HIP__
#define TMPM_BOTH __host__ __device__ __forceinline__
#else
#define TMPM_BOTH inline
#endif

namespace tmpm {

// sqrt(x) for normal x > 0, within an ulp, from y = (1 + e) / sqrt(x) with |e|
// up to 2^-23, which is what v_rsq_f64 is documented to (2^29 ulp).  Each step
// leaves at most 1.5 e times the error before it: 1.2e-7, 2.2e-14, 4e-21 and the
// last rounding.  NaN at 0 (y is infinite).
TMPM_BOTH double refine_root(double x, double y) {
  const double r = x * y, s = __builtin_fma(0.5 * y, __builtin_fma(-r, r, x), r);
  return __builtin_fma(0.5 * y, __builtin_fma(-s, s, x), s);
}

}  // namespace tmpm

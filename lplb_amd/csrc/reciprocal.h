// Reciprocals in fp64 from the hardware's estimate.  No other header here, so that their error can be measured on a CPU with
// an estimate of any error (tests/test_host.py).
#pragma once

namespace lplb {

// 1/a in fp64: hardware estimate (about 2^-23) + one Newton step.
__device__ inline double rcp_f64(double a) {
  double r = __builtin_amdgcn_rcp(a);
  return __builtin_fma(__builtin_fma(-a, r, 1.0), r, r);
}

// 0.999 / d_max in fp64, rounded to fp32 by the caller: estimate, Newton step, one correction of the quotient (one rounding is
// all that is left of its error; the compiler's full division takes twice the instructions, all of them in the chain from one
// step to the next).  Without the Newton step the error would be 2^-46, for 0.013 us a step less at 8 ranks with two slots and
// nothing at 16.  d_max = 0 or infinite gives NaN where the division gives infinity or 0: either way the step leaves the
// artificial variable without a number below the feasibility limit, so the LP is reported infeasible and its shares are the
// neutral ones.
__device__ inline double step_length(double d_max) {
  const double r = rcp_f64(d_max);
  const double q = 0.999 * r;
  return __builtin_fma(__builtin_fma(-d_max, q, 0.999), r, q);
}

} // namespace lplb

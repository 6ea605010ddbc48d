// kde_math.h -- FP64 kernel functions of the evaluation and interpolation
// matrix kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace nck
{

// rsqrt (u) for normal u > 0: the hardware estimate (about 23 good bits)
// and one third-order step.  With e = 1 - u r^2 the exact value is
// r (1 - e)^{-1/2} = r (1 + e / 2 + 3 e^2 / 8 + O(e^3)), and e^3 is below 2^-66.
__device__ inline double
rsqrt_step (double u, double r)
{
  const double e = fma (-(u * r), r, 1.0);

  return fma (r * e, fma (0.375, e, 0.5), r);
}

__device__ inline double
rsqrt_f64 (double u)
{
  return rsqrt_step (u, __builtin_amdgcn_rsq (u));
}

// u^{-p/2} for u >= 1 and a wave-uniform p in [1, 127]: the p-th power of
// rsqrt (u) by squaring (at most 6 squarings and 6 products).  This is the
// Student-t kernel (1 + chi2 / nu)^{-(nu + d) / 2} at integer nu; it costs
// about a fifth of exp (-(nu + d) / 2 log1p (chi2 / nu)), and its relative
// error, p / 2 roundings of u and p of the power, is that of rounding the
// logarithm before the exponential.  Underflows to 0; NaN and inf give NaN.
__device__ inline double
half_power (double u, int p)
{
  double s = rsqrt_f64 (u);
  double t = (p & 1) ? s : 1.0;

#pragma unroll
  for (int bit = 1; bit < 7; ++bit)
  {
    if ((p >> bit) == 0)
      break;

    s = s * s;

    if ((p >> bit) & 1)
      t = t * s;
  }

  return t;
}

// 2^t for t <= 0 (0 below the subnormals): t = n + f with f in [-1/2, 1/2],
// the Taylor polynomial of exp (f ln 2) to order 13 (remainder below
// (ln 2 / 2)^14 / 14! = 5e-18), and the exponent by ldexp.
__device__ inline double
exp2_f64 (double t)
{
  const double n = rint (t);
  const double x = (t - n) * 0.69314718055994530941723212145817657;
  double p       = 1.0 / 6227020800.0;

  p = fma (p, x, 1.0 / 479001600.0);
  p = fma (p, x, 1.0 / 39916800.0);
  p = fma (p, x, 1.0 / 3628800.0);
  p = fma (p, x, 1.0 / 362880.0);
  p = fma (p, x, 1.0 / 40320.0);
  p = fma (p, x, 1.0 / 5040.0);
  p = fma (p, x, 1.0 / 720.0);
  p = fma (p, x, 1.0 / 120.0);
  p = fma (p, x, 1.0 / 24.0);
  p = fma (p, x, 1.0 / 6.0);
  p = fma (p, x, 0.5);
  p = fma (p, x, 1.0);
  p = fma (p, x, 1.0);

  return ldexp (p, (int) n);
}

// Rows of a packed factor that a padded dimension D <= 12 may not need: rows
// from d on are zero and add nothing, so the row loops of the per-pair kernels
// leave at the first even row at or past d above the next smaller dimension.
// (At D = 32 the guards cost more than the rows: the interpolation matrix of
// d = 32, n = 10000 took 8 % longer, since each one ends the scalar loads in
// flight.)
__device__ constexpr bool
row_guard (int D, int r)
{
  return D <= 12 && r > D - 4 && r % 2 == 0;
}

} // namespace nck

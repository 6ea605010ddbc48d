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
// about a fifth of exp (-(nu + d) / 2 log1p (chi2 / nu)).  Its relative error is p / 2
// roundings of u and p of the power, whatever chi2 is; the logarithm's form is
// more accurate near a kernel's centre and less so away from it (largest
// error at nu = 3, power / logarithm: d = 16 2.8e-15 / 1.7e-16 for chi2 below 0.01 d,
// 4.1e-15 / 6.3e-15 from d to 10 d; d = 64 1.1e-14 / 1.2e-15 and 1.5e-14 / 3.1e-14).
// Underflows to 0; NaN and inf give NaN.
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

// a whole number as an int, saturated (-2^31 for -inf, 0 for NaN); outside its
// range the conversion of the language is undefined
__device__ inline int
saturated_int (double n)
{
  int k;

  __asm__ ("v_cvt_i32_f64 %0, %1" : "=v" (k) : "v" (n));

  return k;
}

// S 2^R = the sum of the 2^t that were added (t <= 0), R a whole number up to
// 512 below the largest t: one integer comparison per term instead of a
// maximum and a rescaling, and no term is lost beside a sum of about 1 or more,
// wherever the terms lie.  Terms below 2^-(2^30) add nothing; -inf and NaN make
// the sum NaN.
//
// 2^t is taken as 2^n exp (f ln 2), n = rint (t), f in [-1/2, 1/2].  The
// polynomial 1 + x + x^2 g (x) interpolates g = (exp (x) - 1 - x) / x^2 at the
// Chebyshev nodes of |x| <= ln 2 / 2; its largest error is 3.4e-19 (a Taylor
// polynomial needs one order more for 5e-18).
//
// The rescaling is a wave-uniform branch, kept one by the empty asm: as the
// selects that the compiler makes of it every term pays for it (16 % at d = 4).
// LATE: after the addition, which leaves a step's code in one piece (d = 16, n =
// 4000, m = 20000: 0.79 ms, 0.82 with the branch first), but holds both sums,
// which at d = 64 spills (7.9 against 6.0 ms).
template <bool LATE>
struct Pow2Sum
{
  int R    = -(1 << 30);
  double S = 0.0;

  __device__ inline void
  add (double t)
  {
    const double n = rint (t);
    const double x = (t - n) * 0.69314718055994530941723212145817657;
    int k          = saturated_int (n);
    double p       = 0x1.1f72fc730b4ffp-29;

    p = fma (p, x, 0x1.af4ddd84882fep-26);
    p = fma (p, x, 0x1.27e4db67b4303p-22);
    p = fma (p, x, 0x1.71de02375656cp-19);
    p = fma (p, x, 0x1.a01a01a6d7808p-16);
    p = fma (p, x, 0x1.a01a01abe62ddp-13);
    p = fma (p, x, 0x1.6c16c16c162d6p-10);
    p = fma (p, x, 0x1.11111111100dfp-7);
    p = fma (p, x, 0x1.5555555555556p-5);
    p = fma (p, x, 0x1.5555555555557p-3);
    p = fma (p, x, 0.5);
    p = fma (p, x, 1.0);
    p = fma (p, x, 1.0);

    const double Sn = LATE ? S + ldexp (p, k - R) : 0.0;

    if (__any (k - R > 512))
    {
      __asm__ ("" : "+v" (k));

      const bool up = k - R > 512;
      const int r   = up ? k : R;

      S = (LATE && !up) ? Sn : ldexp (S, R - r) + (LATE ? p : 0.0);
      R = r;
    }
    else if (LATE)
    {
      S = Sn;
    }

    if (!LATE)
      S += ldexp (p, k - R);
  }

  // the sum as s exp (m - ref): with m = ref itself, which every split shares and
  // the merge of the splits takes without an exponential, while s is well
  // within range (R <= 0, since no t is above 0), else with s near 1, so that
  // the larger of two m is that of the larger sum
  __device__ inline void
  result (double ref, double &m, double &s) const
  {
    const int e = __builtin_amdgcn_frexp_exp (S);   // 0 for 0, inf and NaN

    if (R + e > -900)
    {
      m = ref;
      s = ldexp (S, R);
    }
    else
    {
      m = (S > 0.0) ? fma ((double) (R + e), 0.69314718055994530941723212145817657, ref) : -INFINITY;
      s = ldexp (S, -e);
    }
  }
};

// a kernel of [i0, i1) with a weight: a range of zero weights (b = -inf) has
// no terms to form
__device__ inline bool
some_weight (const double *__restrict__ b, int i0, int i1)
{
  bool any = false;

  for (int i = i0; i < i1 && !any; ++i)
    any = (b[i] != -INFINITY);

  return any;
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

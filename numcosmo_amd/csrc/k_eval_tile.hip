// k_eval_tile.hip -- FP64 and FP32 eval of the VKDE from 13 dimensions on,
// with the whitening product on the matrix cores (kde_tile.h).
//
// A wave takes 64 points (FP64 above d = 32: 32) and walks its split's kernels; each lane
// ends a step with the squared norm of one pair and adds its term.  The terms
// and their two forms are those of k_eval.hip, and so are the partial (max,
// sum) pairs that k_eval_merge combines.
#include "kde_math.h"
#include "kde_tile.h"
#include "nckde_internal.h"

namespace nck
{

// the (max, sum) pairs of a point's two lanes, one per kernel of a step
__device__ inline void
join_halves (double &M, double &S)
{
  const double Mo = __shfl_xor (M, 16, 64), So = __shfl_xor (S, 16, 64);
  const double Mx = fmax (M, Mo);

  S = ((M > -INFINITY) ? S * exp (M - Mx) : 0.0) + ((Mo > -INFINITY) ? So * exp (Mo - Mx) : 0.0);
  M = Mx;
}

template <int NK, int KERNEL>
__global__ void __launch_bounds__ (256)
k_eval_tile (EvalArgs a)
{
  typedef PairTile<double, NK> P;
  const int wave  = threadIdx.x >> 6;
  const int p0    = (blockIdx.x * (blockDim.x >> 6) + wave) * P::PTS;
  const int chunk = (a.n + a.nsplit - 1) / a.nsplit;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n, i0 + chunk);

  if (p0 >= a.m)
    return;

  P tile;

  tile.load_points (a.X, p0, a.m, a.d, a.D);

  const int lp = p0 + tile.lane_point ();
  const int lk = tile.lane_kernel ();
  double M     = -INFINITY, S = 0.0;
  bool done    = false;

  // the fast forms of k_eval_f64
  if (KERNEL == NCKDE_KERNEL_GAUSS)
  {
    if (!a.general)
    {
      Pow2Sum<P::KU == 1> sum;

      for (int i = i0; i < i1; i += P::KU)
      {
        const double chi2 = tile.chi2 (a.Wp, a.Th, i, i1);
        const bool on     = (P::KU == 1) || (i + lk < i1);
        const double t    = fma (chi2, a.fc, a.term[on ? i + lk : i]);

        sum.add (on ? t : -1.0e300);
      }

      sum.result (*a.tref, M, S);

      if (P::KU == 2)
        join_halves (M, S);

      done = (S > 0.0) && (S < INFINITY);
    }
  }
  else if (a.pw > 0)
  {
    for (int i = i0; i < i1; i += P::KU)
    {
      const double chi2 = tile.chi2 (a.Wp, a.Th, i, i1);
      const bool on     = (P::KU == 1) || (i + lk < i1);
      const double e    = a.term[on ? i + lk : i] * half_power (fma (chi2, a.fc, 1.0), a.pw);

      S += on ? e : 0.0;
    }

    if (P::KU == 2)
      S += __shfl_xor (S, 16, 64);

    done = (S > EVAL_FAST_FLOOR) && (S < INFINITY);
    M    = *a.tref;
  }

  // the general form, for the wave as long as a lane needs it
  if (__any (!done))
  {
    double Mg = -INFINITY, Sg = 0.0;

    for (int i = some_weight (a.b, i0, i1) ? i0 : i1; i < i1; i += P::KU)
    {
      const double chi2 = tile.chi2 (a.Wp, a.Th, i, i1) * a.inv_h2;
      const bool on     = (P::KU == 1) || (i + lk < i1);
      const double b    = a.b[on ? i + lk : i];
      double lnt;

      if (KERNEL == NCKDE_KERNEL_GAUSS)
        lnt = fma (-0.5, chi2, b);
      else
        lnt = fma (a.kappa, log1p (chi2 / a.nu), b);

      if (!on)
        lnt = -INFINITY;

      if (lnt > Mg)
      {
        Sg = Sg * exp (Mg - lnt);
        Mg = lnt;
      }

      const double e = exp (lnt - Mg);

      Sg += (lnt > -INFINITY) ? e : 0.0;
    }

    if (P::KU == 2)
      join_halves (Mg, Sg);

    if (!done)
    {
      M = Mg;
      S = Sg;
    }
  }

  if (lp < a.m && lk == 0)
  {
    a.partM[(size_t) blockIdx.y * a.m + lp] = M;
    a.partS[(size_t) blockIdx.y * a.m + lp] = S;
  }
}

// the FP32 rung: differences in FP64 rounded to FP32, the product, the norm
// and the kernel in FP32, sums in FP64 (see k_eval_f32)
template <int NK, int KERNEL>
__global__ void __launch_bounds__ (256)
k_eval_tile_f32 (EvalArgs a)
{
  typedef PairTile<float, NK> P;
  const int wave  = threadIdx.x >> 6;
  const int p0    = (blockIdx.x * (blockDim.x >> 6) + wave) * P::PTS;
  const int chunk = (a.n + a.nsplit - 1) / a.nsplit;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n, i0 + chunk);

  if (p0 >= a.m)
    return;

  P tile;

  tile.load_points (a.X, p0, a.m, a.d, a.D);

  const int lp       = p0 + tile.lane_point ();
  const float inv_h2 = (float) a.inv_h2;
  const float kappa  = (float) a.kappa;
  const float inv_nu = (float) (1.0 / a.nu);
  float M            = -INFINITY;
  double S           = 0.0;

  static_assert (P::KU == 1, "one kernel per step");

  for (int i = i0; i < i1; ++i)
  {
    const float chi2 = tile.chi2 (a.Wf, a.Th, i, i1) * inv_h2;
    const float b2   = a.b2f[i];
    float lnt;

    if (KERNEL == NCKDE_KERNEL_GAUSS)
      lnt = fmaf (-0.5f, chi2, b2);
    else
      lnt = fmaf (kappa, log1pf (chi2 * inv_nu), b2);

    if (lnt > M)
    {
      S = S * (double) expf (M - lnt);
      M = lnt;
    }

    S += (lnt > -INFINITY) ? (double) expf (lnt - M) : 0.0;
  }

  if (lp < a.m)
  {
    a.partM[(size_t) blockIdx.y * a.m + lp] = (M > -INFINITY) ? (double) M + a.bref : -INFINITY;
    a.partS[(size_t) blockIdx.y * a.m + lp] = S;
  }
}

template <int NK, int KERNEL>
static hipError_t
tile_t (const EvalArgs &a, hipStream_t s)
{
  const int PTS   = (a.b2f != nullptr) ? PairTile<float, NK>::PTS : PairTile<double, NK>::PTS;
  const int waves = (a.m + PTS - 1) / PTS;
  const int wpb   = (waves < 4) ? waves : 4;
  const dim3 grid ((waves + wpb - 1) / wpb, a.nsplit), block (64 * wpb);

  if (a.b2f != nullptr)
    hipLaunchKernelGGL ((k_eval_tile_f32<NK, KERNEL>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL ((k_eval_tile<NK, KERNEL>), grid, block, 0, s, a);

  return hipGetLastError ();
}

template <int NK>
static hipError_t
tile_k (const EvalArgs &a, hipStream_t s)
{
  return (a.kernel == NCKDE_KERNEL_GAUSS) ? tile_t<NK, NCKDE_KERNEL_GAUSS> (a, s)
                                          : tile_t<NK, NCKDE_KERNEL_ST> (a, s);
}

hipError_t
launch_eval_tile (const EvalArgs &a, hipStream_t s)
{
  switch (tile_nk (a.d))
  {
    case 4: return tile_k<4> (a, s);
    case 5: return tile_k<5> (a, s);
    case 6: return tile_k<6> (a, s);
    case 7: return tile_k<7> (a, s);
    case 8: return tile_k<8> (a, s);
    case 10: return tile_k<10> (a, s);
    case 12: return tile_k<12> (a, s);
    case 14: return tile_k<14> (a, s);
    case 16: return tile_k<16> (a, s);
    default: return hipErrorInvalidValue;
  }
}

} // namespace nck

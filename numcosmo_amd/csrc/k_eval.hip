// k_eval.hip -- FP64 and FP32 eval_m2lnp / eval for KDE, and for VKDE below 13
// dimensions (k_eval_tile.hip has the others).
//
// One lane per evaluation point; every lane of a block walks the same kernel
// range, so the kernel factors (packed W_i = U_i^{-T}, centre, b_i) are
// wave-uniform and come in through scalar loads straight into SGPR operands
// of the FP64 FMAs.  Per pair (VKDE, padded dim D): D subtractions,
// D(D+1)/2 FMAs for z = W_i (x - theta_i), D FMAs for |z|^2, and the kernel's
// term in one of the two forms below.  The kernel range is split over blockIdx.y so that small
// point counts still fill the 256 CUs; partial (max, sum) pairs are merged in
// split order by k_eval_merge.
//
// Reference: ncm_stats_dist_vkde.c:681-723 and ncm_stats_dist_kde.c:639-681
// (eval_weights_m2lnp), the sum0/sum1 reductions of
// ncm_stats_dist_kernel_gauss.c:246-333 / ncm_stats_dist_kernel_st.c:295-386
// and the linear eval_weights (vkde.c:631-679, kde.c:596-637).
#include "kde_math.h"
#include "nckde_internal.h"

namespace nck
{

// The terms are formed in two ways.  Fast: Gauss as 2^t, t relative to max_i
// b_i, summed against a reference that follows the terms (Pow2Sum); Student-t
// with an integer nu up to 127 - d as term_i K against max_i b_i itself, K the
// (nu + d)-th power of an inverse square root.  A lane whose sum is not a
// normal number in range (a point so far out that its terms underflow, NaN or
// inf input) runs the general form instead: ln K with log1p, and an online
// maximum.  The logarithm, the exponential and the maximum of the general form
// cost as much as the 136 FMAs of a d = 16 factor.
//
// A Gauss sum against max_i b_i itself takes 3 % less time on a plain sample,
// but underflows at chi2 = 1150, in every split of other modes, and is not
// finite with a zero weight; it then ran the general form as well (d = 4, n =
// 2000, m = 20000: plain 70 against 73 us here, sorted modes 154 against 74,
// zero weights 155 against 73; the general form alone 94 to 102).
template <int D, int KERNEL, int KIND>
__global__ void __launch_bounds__ (256)
k_eval_f64 (EvalArgs a)
{
  const int p     = blockIdx.x * blockDim.x + threadIdx.x;
  const int chunk = (a.n + a.nsplit - 1) / a.nsplit;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n, i0 + chunk);
  const int pp    = (p < a.m) ? p : (a.m - 1);
  const int d     = a.d;
  const double *xrow = a.X + (size_t) pp * d;
  double x[D];

#pragma unroll
  for (int k = 0; k < D; ++k)
    x[k] = (k < d) ? xrow[k] : 0.0;

  if constexpr (KIND == NCKDE_KDE)
  {
    // v = U_g^{-T} x (gsl_blas_dtrsv Upper/Trans, kde.c:648-652)
    double v[D];

#pragma unroll
    for (int l = 0; l < D; ++l)
    {
      if (l < d)
      {
        double t = x[l];

#pragma unroll
        for (int m = 0; m < l; ++m)
          t = fma (-v[m], a.Ug[m * d + l], t);

        v[l] = t / a.Ug[l * d + l];
      }
      else
      {
        v[l] = 0.0;
      }
    }

#pragma unroll
    for (int l = 0; l < D; ++l)
      x[l] = v[l];
  }

  // |W_i (x - theta_i)|^2, before the bandwidth
  auto chi2_of = [&] (int i) -> double {
    const double *th = a.Th + (size_t) i * D;
    double chi2      = 0.0;

    if (KIND == NCKDE_VKDE)
    {
      const double *W = a.Wp + (size_t) i * (D * (D + 1) / 2);
      double delta[D];

#pragma unroll
      for (int k = 0; k < D; ++k)
        delta[k] = x[k] - th[k];

#pragma unroll
      for (int r = 0; r < D; ++r)
      {
        if (row_guard (D, r) && r >= d)
          break;

        double z = 0.0;

#pragma unroll
        for (int c = 0; c <= r; ++c)
          z = fma (W[r * (r + 1) / 2 + c], delta[c], z);

        chi2 = fma (z, z, chi2);
      }
    }
    else
    {
#pragma unroll
      for (int k = 0; k < D; ++k)
      {
        const double t = th[k] - x[k];

        chi2 = fma (t, t, chi2);
      }
    }

    return chi2;
  };

  double M  = -INFINITY, S = 0.0;
  bool done = false;

  if (KERNEL == NCKDE_KERNEL_GAUSS)
  {
    if (!a.general)
    {
      Pow2Sum<true> sum;

      for (int i = i0; i < i1; ++i)
        sum.add (fma (chi2_of (i), a.fc, a.term[i]));

      sum.result (*a.tref, M, S);
      done = (S > 0.0) && (S < INFINITY);
    }
  }
  else if (a.pw > 0)
  {
    for (int i = i0; i < i1; ++i)
      S = fma (a.term[i], half_power (fma (chi2_of (i), a.fc, 1.0), a.pw), S);

    done = (S > EVAL_FAST_FLOOR) && (S < INFINITY);
    M    = *a.tref;
  }

  if (!done)
  {
    M = -INFINITY;
    S = 0.0;

    for (int i = some_weight (a.b, i0, i1) ? i0 : i1; i < i1; ++i)
    {
      const double chi2 = chi2_of (i) * a.inv_h2;
      double lnt;

      if (KERNEL == NCKDE_KERNEL_GAUSS)
        lnt = fma (-0.5, chi2, a.b[i]);
      else
        lnt = fma (a.kappa, log1p (chi2 / a.nu), a.b[i]);

      if (lnt > M)
      {
        S = S * exp (M - lnt);
        M = lnt;
      }

      {
        const double e = exp (lnt - M);

        S += (lnt > -INFINITY) ? e : 0.0;
      }
    }
  }

  if (p < a.m)
  {
    a.partM[(size_t) blockIdx.y * a.m + p] = M;
    a.partS[(size_t) blockIdx.y * a.m + p] = S;
  }
}

// The FP32 rung of the precision ladder: the same walk in single precision.
// x - theta_i is formed in FP64 and rounded to FP32; W_i comes from its FP32
// copy; |z|^2 and the kernel run in FP32 against a fixed reference,
// lnt = b2_i + ln K with b2_i = b_i - max_j b_j (FP32), with an online FP32
// maximum and the sum in FP64.  The partial maximum is stored back in
// natural units (+ max_j b_j) so that k_eval_merge serves both forms.
template <int D, int KERNEL, int KIND>
__global__ void __launch_bounds__ (256)
k_eval_f32 (EvalArgs a)
{
  const int p     = blockIdx.x * blockDim.x + threadIdx.x;
  const int chunk = (a.n + a.nsplit - 1) / a.nsplit;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n, i0 + chunk);
  const int pp    = (p < a.m) ? p : (a.m - 1);
  const int d     = a.d;
  double x[D];

#pragma unroll
  for (int k = 0; k < D; ++k)
    x[k] = (k < d) ? a.X[(size_t) pp * d + k] : 0.0;

  if (KIND == NCKDE_KDE)
  {
    double v[D];

#pragma unroll
    for (int l = 0; l < D; ++l)
    {
      if (l < d)
      {
        double t = x[l];

#pragma unroll
        for (int m = 0; m < l; ++m)
          t = fma (-v[m], a.Ug[m * d + l], t);

        v[l] = t / a.Ug[l * d + l];
      }
      else
      {
        v[l] = 0.0;
      }
    }

#pragma unroll
    for (int l = 0; l < D; ++l)
      x[l] = v[l];
  }

  const float inv_h2 = (float) a.inv_h2;
  const float kappa  = (float) a.kappa;
  const float inv_nu = (float) (1.0 / a.nu);
  float M            = -INFINITY;
  double S           = 0.0;

  for (int i = i0; i < i1; ++i)
  {
    const double *th = a.Th + (size_t) i * D;
    float chi2       = 0.0f;

    if (KIND == NCKDE_VKDE)
    {
      const float *W = a.Wf + (size_t) i * (D * (D + 1) / 2);
      float delta[D];

#pragma unroll
      for (int k = 0; k < D; ++k)
        delta[k] = (float) (x[k] - th[k]);

#pragma unroll
      for (int r = 0; r < D; ++r)
      {
        float z = 0.0f;

#pragma unroll
        for (int c = 0; c <= r; ++c)
          z = fmaf (W[r * (r + 1) / 2 + c], delta[c], z);

        chi2 = fmaf (z, z, chi2);
      }
    }
    else
    {
#pragma unroll
      for (int k = 0; k < D; ++k)
      {
        const float t = (float) (th[k] - x[k]);

        chi2 = fmaf (t, t, chi2);
      }
    }

    chi2 *= inv_h2;

    float lnt;

    if (KERNEL == NCKDE_KERNEL_GAUSS)
      lnt = fmaf (-0.5f, chi2, a.b2f[i]);
    else
      lnt = fmaf (kappa, log1pf (chi2 * inv_nu), a.b2f[i]);

    if (lnt > M)
    {
      S = S * (double) expf (M - lnt);
      M = lnt;
    }

    S += (lnt > -INFINITY) ? (double) expf (lnt - M) : 0.0;
  }

  if (p < a.m)
  {
    a.partM[(size_t) blockIdx.y * a.m + p] = (M > -INFINITY) ? (double) M + a.bref : -INFINITY;
    a.partS[(size_t) blockIdx.y * a.m + p] = S;
  }
}

// FP32 copies of the packed factors and the shifted b_i
__global__ void
k_f32_factors (const double *__restrict__ Wp, size_t count, float *__restrict__ Wf)
{
  const size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x;

  if (e < count)
    Wf[e] = (float) Wp[e];
}

__global__ void
k_f32_b2 (const double *__restrict__ b, double bref, int n, float *__restrict__ b2f)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;

  if (i < n)
    b2f[i] = (float) (b[i] - bref);
}

hipError_t
launch_f32_factors (const double *Wp, size_t count, float *Wf, hipStream_t s)
{
  if (count > 0)
    hipLaunchKernelGGL (k_f32_factors, dim3 ((unsigned) ((count + 255) / 256)), dim3 (256), 0, s, Wp, count, Wf);

  return hipGetLastError ();
}

hipError_t
launch_f32_b2 (const double *b, double bref, int n, float *b2f, hipStream_t s)
{
  hipLaunchKernelGGL (k_f32_b2, dim3 ((n + 255) / 256), dim3 (256), 0, s, b, bref, n, b2f);

  return hipGetLastError ();
}

// gamma = max over splits, S = sum_s S_s exp(M_s - gamma);
// m2lnp = -2 (gamma - lnnorm_shared + ln S - d ln h)
//
// A block takes 256 / L points with L lanes each.  Lane l takes the splits l,
// l + L, ...; the lanes' maxima and sums combine as a tree in LDS, so the
// result depends on nsplit and L only.  The reads of the partials bound it:
// 8 lanes keep 256-byte rows coalesced over 32 points and are used from 2048
// points on; below, 64 lanes (256 up to 256 points) shorten the serial walk
// over the splits, which one lane per point ran in 66 us at m = 6400.
__global__ void __launch_bounds__ (256)
k_eval_merge (EvalArgs a, int L)
{
  __shared__ double red[256];
  const int np = 256 / L;
  const int pl = threadIdx.x % np, sl = threadIdx.x / np;
  const int p  = blockIdx.x * np + pl;
  const int pp = (p < a.m) ? p : a.m - 1;
  double M     = -INFINITY;

  for (int s = sl; s < a.nsplit; s += L)
    M = fmax (M, a.partM[(size_t) s * a.m + pp]);

  red[threadIdx.x] = M;
  __syncthreads ();

  for (int o = L / 2; o > 0; o >>= 1)
  {
    if (sl < o)
      red[threadIdx.x] = fmax (red[threadIdx.x], red[threadIdx.x + o * np]);

    __syncthreads ();
  }

  M = red[pl];
  __syncthreads ();

  double S = 0.0;

  for (int s = sl; s < a.nsplit; s += L)
  {
    const double Ms = a.partM[(size_t) s * a.m + pp];
    const double Ss = a.partS[(size_t) s * a.m + pp];

    if (Ms == M)
      S += (M > -INFINITY) ? Ss : 0.0;
    else if (Ms > -INFINITY)
      S += Ss * exp (Ms - M);
  }

  red[threadIdx.x] = S;
  __syncthreads ();

  for (int o = L / 2; o > 0; o >>= 1)
  {
    if (sl < o)
      red[threadIdx.x] += red[threadIdx.x + o * np];

    __syncthreads ();
  }

  if (sl != 0 || p >= a.m)
    return;

  const double m2lnp = -2.0 * ((M - a.lnnorm_shared) + log (red[pl]) - a.lnh_d);

  a.out[p] = a.linear ? exp (-0.5 * m2lnp) : m2lnp;
}

// The per-kernel constants of the fast form against bref = max_i b_i:
// Student-t term_i = exp (b_i - bref), Gauss term_i = (b_i - bref) log2 e, and
// -1e300 for a zero weight (finite, and below every sum's range); term[n] =
// bref.  One block: the arrays are n doubles.
__global__ void __launch_bounds__ (1024)
k_eval_terms (const double *__restrict__ b, int n, int kernel, double *__restrict__ term,
              const int *__restrict__ status)
{
  __shared__ double red[1024];
  double M = -INFINITY;

  if (status != nullptr && *status != 0)
    return;

  for (int i = threadIdx.x; i < n; i += 1024)
    M = fmax (M, b[i]);

  red[threadIdx.x] = M;
  __syncthreads ();

  for (int o = 512; o > 0; o >>= 1)
  {
    if (threadIdx.x < o)
      red[threadIdx.x] = fmax (red[threadIdx.x], red[threadIdx.x + o]);

    __syncthreads ();
  }

  M = red[0];

  for (int i = threadIdx.x; i < n; i += 1024)
  {
    const double t = b[i] - M;

    term[i] = (kernel != NCKDE_KERNEL_GAUSS) ? exp (t) : (t == -INFINITY) ? -1.0e300 : t * LOG2E_D;
  }

  if (threadIdx.x == 0)
    term[n] = M;
}

hipError_t
launch_eval_terms (const double *b, int n, int kernel, double *term, const int *status, hipStream_t s)
{
  hipLaunchKernelGGL (k_eval_terms, dim3 (1), dim3 (1024), 0, s, b, n, kernel, term, status);

  return hipGetLastError ();
}

template <int D, int KERNEL, int KIND>
static hipError_t
launch_t (const EvalArgs &a, hipStream_t s)
{
  // one wave holds up to 64 points: further waves of a block would repeat it
  const int bs = (a.m <= 64) ? 64 : (a.m <= 128) ? 128 : 256;
  dim3 grid ((a.m + bs - 1) / bs, a.nsplit);

  if (a.b2f != nullptr)
    hipLaunchKernelGGL ((k_eval_f32<D, KERNEL, KIND>), grid, dim3 (bs), 0, s, a);
  else
    hipLaunchKernelGGL ((k_eval_f64<D, KERNEL, KIND>), grid, dim3 (bs), 0, s, a);

  return hipGetLastError ();
}

template <int D>
static hipError_t
launch_d (const EvalArgs &a, hipStream_t s)
{
  if constexpr (D < TILE_MIN_D)
    if (a.kind == NCKDE_VKDE)
      return (a.kernel == NCKDE_KERNEL_GAUSS) ? launch_t<D, NCKDE_KERNEL_GAUSS, NCKDE_VKDE> (a, s)
                                              : launch_t<D, NCKDE_KERNEL_ST, NCKDE_VKDE> (a, s);

  return (a.kernel == NCKDE_KERNEL_GAUSS) ? launch_t<D, NCKDE_KERNEL_GAUSS, NCKDE_KDE> (a, s)
                                          : launch_t<D, NCKDE_KERNEL_ST, NCKDE_KDE> (a, s);
}

int
padded_dim (int d)
{
  static const int dims[] = {4, 8, 12, 16, 24, 32, 48, 64};

  for (int D : dims)
    if (d <= D)
      return D;

  return -1;
}

hipError_t
launch_eval_f64 (const EvalArgs &a, hipStream_t s)
{
  if (a.kind == NCKDE_VKDE && a.d >= TILE_MIN_D)
    return launch_eval_tile (a, s);

  switch (a.D)
  {
    case 4: return launch_d<4> (a, s);
    case 8: return launch_d<8> (a, s);
    case 12: return launch_d<12> (a, s);
    case 16: return launch_d<16> (a, s);
    case 24: return launch_d<24> (a, s);
    case 32: return launch_d<32> (a, s);
    case 48: return launch_d<48> (a, s);
    case 64: return launch_d<64> (a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t
launch_eval_merge (const EvalArgs &a, hipStream_t s)
{
  const int L = (a.m >= 2048) ? 8 : (a.m > 256) ? 64 : 256;

  hipLaunchKernelGGL (k_eval_merge, dim3 ((a.m + 256 / L - 1) / (256 / L)), dim3 (256), 0, s, a, L);

  return hipGetLastError ();
}

} // namespace nck

// k_im_tile.hip -- interpolation matrix of the VKDE from 13 dimensions on,
// with the whitening product on the matrix cores (kde_tile.h).
//
// A[j][i] = K(chi2_ij) / (u_i h^d) / f_j as in k_build_IM (k_linalg.hip),
// whose kernel expressions and normalisation staging it shares; a wave takes
// 64 (or 32) observations and stores whole 512- (or 128-) byte rows of A^T.
#include "kde_math.h"
#include "kde_tile.h"
#include "nckde_internal.h"

namespace nck
{

constexpr int IMT_KB = 256;   // kernels whose normalisation a block forms at a time

template <int NK, int KERNEL>
__global__ void __launch_bounds__ (256)
k_im_tile (IMArgs a, const double *__restrict__ Wp, const double *__restrict__ Th, double *__restrict__ AT)
{
  typedef PairTile<double, NK> P;
  __shared__ double kscale[IMT_KB];
  const int wave  = threadIdx.x >> 6;
  const int p0    = (blockIdx.x * 4 + wave) * P::PTS;
  const int chunk = (a.n_k + gridDim.y - 1) / gridDim.y;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n_k, i0 + chunk);
  P tile;

  // waves past the last observation repeat it and store nothing
  tile.load_points (a.X, p0, a.n_obs, a.d, a.D);

  const int j  = p0 + tile.lane_point ();
  const int jj = min (j, a.n_obs - 1);
  const int lk = tile.lane_kernel ();

  double rowscale = 1.0;

  if (a.m2lnp)
    rowscale = 1.0 / exp (-0.5 * (a.m2lnp[jj] - a.min_m2lnp));

  const double kappa  = -0.5 * (a.nu + (double) (unsigned) a.d);
  const double inv_nu = 1.0 / a.nu;

  for (int ib = i0; ib < i1; ib += IMT_KB)
  {
    const int ie = min (i1, ib + IMT_KB);

    __syncthreads ();

    if (ib + (int) threadIdx.x < ie)
      kscale[threadIdx.x] = 1.0 / exp (a.lnnorm[ib + threadIdx.x] + a.lnnorm_href);

    __syncthreads ();

    for (int i = ib; i < ie; i += P::KU)
    {
      const double chi2 = tile.chi2 (Wp, Th, i, ie) * a.inv_h2;
      const double u    = fma (chi2, inv_nu, 1.0);
      double K;

      if (KERNEL == NCKDE_KERNEL_GAUSS)
        K = exp (-0.5 * chi2);
      else if (a.pw > 0 && u < 1.0e290)
        K = half_power (u, a.pw);
      else
        K = exp (kappa * log1p (chi2 * inv_nu));

      if (j < a.n_obs && i + lk < ie)
        AT[(size_t) (i + lk) * a.n_obs + j] = (K * kscale[i + lk - ib]) * rowscale;
    }
  }
}

// the grid of k_build_IM: about 2048 blocks in whole rounds of the blocks the
// device holds at once
template <int NK, int KERNEL>
static hipError_t
imt_t (const IMArgs &a, hipStream_t s)
{
  static const int resident = [] {
    int dev = 0, ncu = 0, nb = 0;

    (void) hipGetDevice (&dev);
    (void) hipDeviceGetAttribute (&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    (void) hipOccupancyMaxActiveBlocksPerMultiprocessor (&nb, k_im_tile<NK, KERNEL>, 256, 0);
    return (nb > 0 ? nb : 1) * (ncu > 0 ? ncu : 1);
  }();

  constexpr int PB = 4 * PairTile<double, NK>::PTS;
  const int bx     = (a.n_obs + PB - 1) / PB;
  const int total0 = bx * ((2048 + bx - 1) / bx);
  const int rounds = (total0 + resident / 2) / resident;
  int gy           = (rounds > 0 ? rounds : 1) * resident / bx;

  gy = (gy > a.n_k) ? a.n_k : gy;
  gy = (gy < 1) ? 1 : gy;

  hipLaunchKernelGGL ((k_im_tile<NK, KERNEL>), dim3 (bx, gy), dim3 (256), 0, s, a, a.Wp, a.Th, a.AT);

  return hipGetLastError ();
}

template <int NK>
static hipError_t
imt_k (const IMArgs &a, hipStream_t s)
{
  return (a.kernel == NCKDE_KERNEL_GAUSS) ? imt_t<NK, NCKDE_KERNEL_GAUSS> (a, s) : imt_t<NK, NCKDE_KERNEL_ST> (a, s);
}

hipError_t
launch_im_tile (const IMArgs &a, hipStream_t s)
{
  switch (tile_nk (a.d))
  {
    case 4: return imt_k<4> (a, s);
    case 5: return imt_k<5> (a, s);
    case 6: return imt_k<6> (a, s);
    case 7: return imt_k<7> (a, s);
    case 8: return imt_k<8> (a, s);
    case 10: return imt_k<10> (a, s);
    case 12: return imt_k<12> (a, s);
    case 14: return imt_k<14> (a, s);
    case 16: return imt_k<16> (a, s);
    default: return hipErrorInvalidValue;
  }
}

} // namespace nck

// k_linalg.hip -- interpolation matrix and the FP64 linear algebra of the
// active-set NNLS weight fit.
//
// The interpolation matrix is stored column-major, AT[i][j] = A[j][i]
// (kernel i, observation j), so that building it, scaling its rows and both
// matrix-vector products of the NNLS loop read and write unit-stride rows.
//
// Reference: _ncm_stats_dist_compute_IM_full (ncm_stats_dist.c:791-804),
// compute_IM (ncm_stats_dist_kde.c:492-557, ncm_stats_dist_vkde.c:517-606),
// ncm_nnls_solve and its normal-equation solvers (ncm_nnls.c:464-871).
#include "kde_math.h"
#include "nckde_internal.h"

namespace nck
{

// --------------------------------------------------------------------------
// A[j][i] = K(chi2_ij) / (u_i h^d) / f_j,  f_j = exp(-(m2lnp_j - min)/2)
// One thread per observation j, a block per (256 observations, kernel
// chunk).  The per-kernel normalisation 1 / exp(lnnorm_i + d ln h) is formed
// once per block for 256 kernels at a time in LDS, and the Student-t kernel
// is exp(kappa log1p(chi2 / nu)) (equal to the reference's pow form to a few
// ulp).  Threads past the last observation take part in the LDS staging only.
// --------------------------------------------------------------------------
constexpr int IM_KB = 256;

// The kernel factors come through scalar loads only when the compiler knows
// that the stores into AT cannot reach them: hence the separate __restrict__
// arguments (with the pointers inside IMArgs the loop loaded every factor
// entry with vector loads and waited on each, 3x slower).
template <int D, int KERNEL, int KIND>
__global__ void __launch_bounds__ (256)
k_build_IM (IMArgs a, const double *__restrict__ Wp, const double *__restrict__ Th, double *__restrict__ AT)
{
  __shared__ double kscale[IM_KB];
  const int j     = blockIdx.x * 256 + threadIdx.x;
  const int chunk = (a.n_k + gridDim.y - 1) / gridDim.y;
  const int i0    = blockIdx.y * chunk;
  const int i1    = min (a.n_k, i0 + chunk);
  const bool live = (j < a.n_obs);
  const int jj    = live ? j : (a.n_obs - 1);
  const int d     = a.d;
  // at D >= 32 the point is read again for every kernel (from L1/L2) instead
  // of being held in registers beside the differences
  constexpr bool XREG = (D < 32);
  const double *xrow  = ((KIND == NCKDE_VKDE) ? a.X : a.Y) + (size_t) jj * d;
  double xj[XREG ? D : 1];

  if (XREG)
  {
#pragma unroll
    for (int k = 0; k < D; ++k)
      xj[k] = (k < d) ? xrow[k] : 0.0;
  }

  double rowscale = 1.0;

  if (a.m2lnp)
    rowscale = 1.0 / exp (-0.5 * (a.m2lnp[jj] - a.min_m2lnp));

  const double kappa  = -0.5 * (a.nu + (double) (unsigned) d);
  const double inv_nu = 1.0 / a.nu;

  for (int ib = i0; ib < i1; ib += IM_KB)
  {
    const int ie = min (i1, ib + IM_KB);

    if (KIND == NCKDE_VKDE)
    {
      __syncthreads ();

      if (ib + (int) threadIdx.x < ie)
        kscale[threadIdx.x] = 1.0 / exp (a.lnnorm[ib + threadIdx.x] + a.lnnorm_href);

      __syncthreads ();
    }

    if (!live)
      continue;

    for (int i = ib; i < ie; ++i)
    {
      const double *th = Th + (size_t) i * D;
      double chi2      = 0.0;
      double scale;

      if (KIND == NCKDE_VKDE)
      {
        const double *W = Wp + (size_t) i * (D * (D + 1) / 2);
        double delta[D];

#pragma unroll
        for (int k = 0; k < D; ++k)
          delta[k] = (XREG ? xj[k] : ((k < d) ? xrow[k] : 0.0)) - th[k];

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

        chi2  = chi2 * a.inv_h2;
        scale = kscale[i - ib];
      }
      else
      {
#pragma unroll
        for (int k = 0; k < D; ++k)
        {
          const double t = th[k] - (XREG ? xj[k] : ((k < d) ? xrow[k] : 0.0));

          chi2 = fma (t, t, chi2);
        }

        chi2  = chi2 * a.inv_h2;
        scale = a.kde_scale;
      }

      double K;

      const double u = fma (chi2, inv_nu, 1.0);

      if (KERNEL == NCKDE_KERNEL_GAUSS)
        K = exp (-0.5 * chi2);
      else if (a.pw > 0 && u < 1.0e290)
        K = half_power (u, a.pw);
      else
        K = exp (kappa * log1p (chi2 * inv_nu));

      AT[(size_t) i * a.n_obs + j] = (K * scale) * rowscale;
    }
  }
}

// Grid: about 2048 blocks, rounded to whole rounds of the blocks the device
// holds at once, so that no nearly empty last round doubles a block's time
// (n_obs = 3200: 2054 blocks were 2 rounds and 6 blocks).
template <int D, int KERNEL, int KIND>
static hipError_t
im_t (const IMArgs &a, hipStream_t s)
{
  static const int resident = [] {
    int dev = 0, ncu = 0, nb = 0;

    (void) hipGetDevice (&dev);
    (void) hipDeviceGetAttribute (&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    (void) hipOccupancyMaxActiveBlocksPerMultiprocessor (&nb, k_build_IM<D, KERNEL, KIND>, 256, 0);
    return (nb > 0 ? nb : 1) * (ncu > 0 ? ncu : 1);
  }();

  const int bx     = (a.n_obs + 255) / 256;
  const int total0 = bx * ((2048 + bx - 1) / bx);
  const int rounds = (total0 + resident / 2) / resident;
  int gy           = (rounds > 0 ? rounds : 1) * resident / bx;

  if (gy > a.n_k)
    gy = a.n_k;

  if (gy < 1)
    gy = 1;

  hipLaunchKernelGGL ((k_build_IM<D, KERNEL, KIND>), dim3 (bx, gy), dim3 (256), 0, s, a, a.Wp, a.Th, a.AT);

  return hipGetLastError ();
}

template <int D>
static hipError_t
im_d (const IMArgs &a, hipStream_t s)
{
  if constexpr (D < TILE_MIN_D)
    if (a.kind == NCKDE_VKDE)
      return (a.kernel == NCKDE_KERNEL_GAUSS) ? im_t<D, NCKDE_KERNEL_GAUSS, NCKDE_VKDE> (a, s)
                                              : im_t<D, NCKDE_KERNEL_ST, NCKDE_VKDE> (a, s);

  return (a.kernel == NCKDE_KERNEL_GAUSS) ? im_t<D, NCKDE_KERNEL_GAUSS, NCKDE_KDE> (a, s)
                                          : im_t<D, NCKDE_KERNEL_ST, NCKDE_KDE> (a, s);
}

hipError_t
launch_build_IM (const IMArgs &a, hipStream_t s)
{
  if (a.kind == NCKDE_VKDE && a.d >= TILE_MIN_D)
    return launch_im_tile (a, s);

  switch (a.D)
  {
    case 4: return im_d<4> (a, s);
    case 8: return im_d<8> (a, s);
    case 12: return im_d<12> (a, s);
    case 16: return im_d<16> (a, s);
    case 24: return im_d<24> (a, s);
    case 32: return im_d<32> (a, s);
    case 48: return im_d<48> (a, s);
    case 64: return im_d<64> (a, s);
    default: return hipErrorInvalidValue;
  }
}

// out[c][r] = in[r][c]
__global__ void
k_transpose (const double *__restrict__ in, int rows, int cols, double *__restrict__ out)
{
  __shared__ double tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x, ty = threadIdx.y;

  for (int k = ty; k < 32; k += 8)
  {
    const int r = r0 + k, c = c0 + tx;

    tile[k][tx] = (r < rows && c < cols) ? in[(size_t) r * cols + c] : 0.0;
  }

  __syncthreads ();

  for (int k = ty; k < 32; k += 8)
  {
    const int c = c0 + k, r = r0 + tx;

    if (r < rows && c < cols)
      out[(size_t) c * rows + r] = tile[tx][k];
  }
}

hipError_t
launch_transpose (const double *in, int rows, int cols, double *out, hipStream_t s)
{
  dim3 grid ((cols + 31) / 32, (rows + 31) / 32);

  hipLaunchKernelGGL (k_transpose, grid, dim3 (32, 8), 0, s, in, rows, cols, out);

  return hipGetLastError ();
}

// --------------------------------------------------------------------------
// Symmetric rank-K products on the FP64 matrix cores (v_mfma_f64_16x16x4f64)
// over BM x BM tiles of the upper triangle.  256 threads = 4 waves in a
// 2 x 2 layout, each wave a BM/2 x BM/2 block of 16 x 16 MFMA tiles; K
// staged through LDS in slices of 16, the next slice's global loads in
// flight during the current slice's MFMAs.  k_gram forms the Gram matrix of
// the normal equations, k_syrk_mfma the trailing update of the Cholesky's
// super-panels (k_potrf.hip): S[a][b] -= sum_r S[kb+r][a] S[kb+r][b] over the
// rows kb..kb+K-1, for off <= a <= b (upper triangle only).
// Tiles are numbered along the rows of the upper triangle; the grid is
// padded to a multiple of 8 and block b takes tile (b % 8) * (grid / 8) +
// b / 8, so that each XCD (blocks are dealt round-robin over the 8 XCDs)
// works on a contiguous band of tiles that shares operand rows in its L2.
// --------------------------------------------------------------------------
typedef double f64x4 __attribute__ ((ext_vector_type (4)));

constexpr int SY_BK = 16;

// BM: square tile of one block (128 or 64); every thread stages
// VPT = 16 BM / 256 values of each operand per K slice, 16 threads per K row
template <int BM>
__device__ inline void
syrk_load (const double *__restrict__ P, int n, int K, int ld, int kb, int r0, int k0, double (&v)[BM / 16])
{
  constexpr int VPT = BM / 16;
  const int tid     = threadIdx.x;

  const int kq = k0 + tid / 16;
  const int a  = r0 + (tid % 16) * VPT;

#pragma unroll
  for (int q = 0; q < VPT; ++q)
    v[q] = (a + q < n && kq < K) ? P[(size_t) (kb + kq) * ld + a + q] : 0.0;
}

template <int BM>
__device__ inline void
syrk_store (double (*T)[BM + 4], const double (&v)[BM / 16])
{
  constexpr int VPT = BM / 16;
  const int tid     = threadIdx.x;

  const int kk = tid / 16, rr = (tid % 16) * VPT;

#pragma unroll
  for (int q = 0; q < VPT; ++q)
    T[kk][rr + q] = v[q];
}

template <int BM>
__global__ void __launch_bounds__ (256)
k_syrk_mfma (const double *__restrict__ P, int n, int K, int ld, int off, int kb, double *__restrict__ M,
             int ntiles)
{
  static_assert (BM == 128 || BM == 64, "128- or 64-wide tiles");
  constexpr int WM = BM / 2;    // tile of one wave
  constexpr int NI = WM / 16;   // 16 x 16 MFMA blocks per wave dimension

  __shared__ double As[SY_BK][BM + 4];
  __shared__ double Bs[SY_BK][BM + 4];

  const int per = gridDim.x / 8;
  int t         = (blockIdx.x % 8) * per + blockIdx.x / 8;

  if (t >= ntiles)
    return;

  const int nt = (n - off + BM - 1) / BM;
  int ti       = 0;

  while (t >= nt - ti)
  {
    t -= nt - ti;
    ++ti;
  }

  const int tj   = ti + t;
  const int r0   = off + ti * BM, c0 = off + tj * BM;
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const int wr   = (w >> 1) * WM, wc = (w & 1) * WM;
  const int li   = lane % 16, lk = lane / 16;

  f64x4 acc[NI][NI];

#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

  double va[BM / 16], vb[BM / 16];

  syrk_load<BM> (P, n, K, ld, kb, r0, 0, va);
  syrk_load<BM> (P, n, K, ld, kb, c0, 0, vb);

  for (int k0 = 0; k0 < K; k0 += SY_BK)
  {
    __syncthreads ();
    syrk_store<BM> (As, va);
    syrk_store<BM> (Bs, vb);
    __syncthreads ();

    if (k0 + SY_BK < K)
    {
      syrk_load<BM> (P, n, K, ld, kb, r0, k0 + SY_BK, va);
      syrk_load<BM> (P, n, K, ld, kb, c0, k0 + SY_BK, vb);
    }

#pragma unroll
    for (int ks = 0; ks < SY_BK / 4; ++ks)
    {
      const int kq = ks * 4 + lk;
      double fa[NI], fb[NI];

#pragma unroll
      for (int i = 0; i < NI; ++i)
      {
        fa[i] = As[kq][wr + i * 16 + li];
        fb[i] = Bs[kq][wc + i * 16 + li];
      }

#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64 (fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  }

  // D[i][j] of a 16 x 16 tile: register r of a lane holds i = lane / 16 + 4 r, j = lane % 16
  // read-modify-write of the tile, one 16-column block at a time with all
  // loads of a lane in flight (out-of-range entries read element 0)
#pragma unroll
  for (int j = 0; j < NI; ++j)
  {
    const int b = c0 + wc + j * 16 + li;
    double old[NI][4];

#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
      {
        const int a  = r0 + wr + i * 16 + lk + 4 * r;
        const bool v = (a < n && b < n && a <= b);

        old[i][r] = M[v ? (size_t) a * ld + b : 0];
      }

#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
      {
        const int a = r0 + wr + i * 16 + lk + 4 * r;

        if (a < n && b < n && a <= b)
          M[(size_t) a * ld + b] = old[i][r] - acc[i][j][r];
      }
  }
}

// Gram matrix M = AT AT^T (AT is n x K row-major): A^T A of the NNLS normal
// equations (cblas_dsyrk, ncm_matrix.c:1547-1575), both triangles written.
// Slices of 16 columns in two LDS buffers, one barrier per slice, the next
// slice's loads in flight under the MFMAs; 16 threads read a row's 128 bytes,
// which stays coalesced for odd K.  n = 10000: 18.4 -> 17.4 ms, n = 2503: 0.46
// -> 0.39 ms against the transposing stage of k_syrk_mfma (57 TFLOP/s of a
// library GEMM's 72).
template <int BM>
__global__ void __launch_bounds__ (256)
k_gram (const double *__restrict__ P, int n, int K, double *__restrict__ M, int ntiles)
{
  static_assert (BM == 128 || BM == 64, "128- or 64-wide tiles");
  constexpr int WM = BM / 2, NI = WM / 16;      // tile of one wave, its 16 x 16 MFMA blocks per dimension
  constexpr int BK = SY_BK, LD = BK + 2;        // row stride in LDS: 16 rows x 4 columns hit every bank once per cycle
  constexpr int RPT = 256 / BK, VPT = BM / RPT; // staged rows per pass, entries per thread
  __shared__ double As[2][BM][LD];
  __shared__ double Bs[2][BM][LD];
  const int per = gridDim.x / 8;
  int t         = (blockIdx.x % 8) * per + blockIdx.x / 8;

  if (t >= ntiles)
    return;

  const int nt = (n + BM - 1) / BM;
  int ti       = 0;

  while (t >= nt - ti)
  {
    t -= nt - ti;
    ++ti;
  }

  const int r0   = ti * BM, c0 = (ti + t) * BM;
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const int wr   = (w >> 1) * WM, wc = (w & 1) * WM;
  const int li   = lane % 16, lk = lane / 16;
  const int sk   = threadIdx.x % BK, sr = threadIdx.x / BK;
  const double *pa[VPT], *pb[VPT];
  f64x4 acc[NI][NI];

#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

  double va[VPT], vb[VPT];

  // rows past n repeat the last one (their products are not stored)
#pragma unroll
  for (int q = 0; q < VPT; ++q)
  {
    pa[q] = P + (size_t) min (r0 + sr + RPT * q, n - 1) * K;
    pb[q] = P + (size_t) min (c0 + sr + RPT * q, n - 1) * K;
  }

  auto load = [&] (int k0) {
    const int k   = k0 + sk;
    const bool in = k < K;
    const int kk  = in ? k : K - 1;

#pragma unroll
    for (int q = 0; q < VPT; ++q)
    {
      va[q] = pa[q][kk];
      vb[q] = pb[q][kk];
    }

    if (!in)
    {
#pragma unroll
      for (int q = 0; q < VPT; ++q)
        va[q] = vb[q] = 0.0;
    }
  };
  auto store = [&] (int b) {
#pragma unroll
    for (int q = 0; q < VPT; ++q)
    {
      As[b][sr + RPT * q][sk] = va[q];
      Bs[b][sr + RPT * q][sk] = vb[q];
    }
  };

  load (0);
  store (0);
  __syncthreads ();

  int cur = 0;

  for (int k0 = 0; k0 < K; k0 += BK)
  {
    if (k0 + BK < K)
      load (k0 + BK);

#pragma unroll
    for (int ks = 0; ks < BK / 4; ++ks)
    {
      double fa[NI], fb[NI];

#pragma unroll
      for (int i = 0; i < NI; ++i)
      {
        fa[i] = As[cur][wr + i * 16 + li][4 * ks + lk];
        fb[i] = Bs[cur][wc + i * 16 + li][4 * ks + lk];
      }

#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64 (fa[i], fb[j], acc[i][j], 0, 0, 0);
    }

    if (k0 + BK < K)
      store (cur ^ 1);

    cur ^= 1;
    __syncthreads ();
  }

#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
      {
        const int a = r0 + wr + i * 16 + lk + 4 * r;
        const int b = c0 + wc + j * 16 + li;

        if (a < n && b < n && a <= b)
        {
          M[(size_t) a * n + b] = acc[i][j][r];
          M[(size_t) b * n + a] = acc[i][j][r];
        }
      }
}

template <int BM>
static void
launch_syrk_mfma (const double *P, int n, int K, int ld, int off, int kb, double *M, hipStream_t s)
{
  const int nt     = (n - off + BM - 1) / BM;
  const int ntiles = nt * (nt + 1) / 2;
  const int grid   = (ntiles + 7) / 8 * 8;

  if (ntiles > 0)
    hipLaunchKernelGGL ((k_syrk_mfma<BM>), dim3 (grid), dim3 (256), 0, s, P, n, K, ld, off, kb, M, ntiles);
}

template <int BM>
static void
gram_t (const double *AT, int n, int K, double *M, hipStream_t s)
{
  const int nt     = (n + BM - 1) / BM;
  const int ntiles = nt * (nt + 1) / 2;

  hipLaunchKernelGGL (k_gram<BM>, dim3 ((ntiles + 7) / 8 * 8), dim3 (256), 0, s, AT, n, K, M, ntiles);
}

hipError_t
launch_gram_nt (const double *AT, int n, int K, double *M, hipStream_t s)
{
  // 128-wide tiles reuse each staged operand twice as often; below about seven
  // blocks per CU their tail leaves the chip half idle, and 64-wide tiles (4x
  // the blocks) balance better (128- against 64-wide: n = 5800 4.3 / 4.0 ms, 6400
  // and 7000 equal, 7600 8.1 / 8.6, 8800 11.8 / 13.4, 10000 18.3 / 19.5)
  const int nt128 = (n + 127) / 128;

  if (nt128 * (nt128 + 1) / 2 >= 1800)
    gram_t<128> (AT, n, K, M, s);
  else
    gram_t<64> (AT, n, K, M, s);

  return hipGetLastError ();
}

// Row sums of IM for the leave-one-out criteria (ncm_stats_dist.c:512-600):
// thread j walks the kernels i = 0..nk-1 of observation j in ascending order,
// the order of the reference's row loops, skipping i == j; the loads go out
// in batches of 16 so that they overlap.
__global__ void
k_im_obs_sums (const double *__restrict__ AT, int nk, int nobs, double *__restrict__ off, double *__restrict__ diag)
{
  const int j = blockIdx.x * blockDim.x + threadIdx.x;

  if (j >= nobs)
    return;

  double s = 0.0;
  int i    = 0;

  for (; i + 16 <= nk; i += 16)
  {
    double v[16];

#pragma unroll
    for (int q = 0; q < 16; ++q)
      v[q] = AT[(size_t) (i + q) * nobs + j];

#pragma unroll
    for (int q = 0; q < 16; ++q)
      s += (i + q != j) ? v[q] : 0.0;
  }

  for (; i < nk; ++i)
    s += (i != j) ? AT[(size_t) i * nobs + j] : 0.0;

  off[j]  = s;
  diag[j] = (j < nk) ? AT[(size_t) j * nobs + j] : 0.0;
}

hipError_t
launch_im_obs_sums (const double *AT, int nk, int nobs, double *off, double *diag, hipStream_t s)
{
  if (nobs > 0)
    hipLaunchKernelGGL (k_im_obs_sums, dim3 ((nobs + 127) / 128), dim3 (128), 0, s, AT, nk, nobs, off, diag);

  return hipGetLastError ();
}

// out[a] = sum_j AT[a][j] v[j] (v == NULL: ones).  One wave per row.
__global__ void
k_row_dot (const double *__restrict__ AT, int n, int K, const double *__restrict__ v, double *__restrict__ out)
{
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / 64;
  const int lane = threadIdx.x % 64;

  if (wave >= n)
    return;

  const double *row = AT + (size_t) wave * K;
  double s          = 0.0;

  for (int j = lane; j < K; j += 64)
    s = fma (row[j], v ? v[j] : 1.0, s);

  for (int o = 32; o > 0; o >>= 1)
    s += __shfl_xor (s, o, 64);

  if (lane == 0)
    out[wave] = s;
}

hipError_t
launch_row_dot (const double *AT, int n, int K, const double *v, double *out, hipStream_t s)
{
  hipLaunchKernelGGL (k_row_dot, dim3 ((n + 3) / 4), dim3 (256), 0, s, AT, n, K, v, out);

  return hipGetLastError ();
}

// r = f - A x (f == NULL: ones) and |r|^2.  Pass 1: block (jb, c) sums the
// kernels of chunk c (res_chunk kernels, inactive ones skipped: x is uniform
// over the block) for 256 observations; pass 2 adds the chunks in a fixed
// order and forms per-block partial sums of r^2; a last pass adds those.
// Chunks: about 2048 blocks in all, at most 4096 chunks (n = 3200: 21
// kernels per chunk; 512-kernel chunks left 91 blocks whose threads each ran
// a 512-step serial chain, 188 us).
static int
res_chunk (int nk, int nobs)
{
  const int nb = (nobs + 255) / 256;
  int nch      = (2048 + nb - 1) / nb;

  nch = (nch < 1) ? 1 : ((nch > 4096) ? 4096 : nch);
  nch = (nch > nk) ? nk : nch;

  return (nk + nch - 1) / (nch > 0 ? nch : 1);
}

__global__ void __launch_bounds__ (256)
k_residual_part (const double *__restrict__ AT, int nk, int nobs, const double *__restrict__ x, int ch,
                 double *__restrict__ part)
{
  const int j  = blockIdx.x * 256 + threadIdx.x;
  const int a0 = blockIdx.y * ch;
  const int a1 = (a0 + ch < nk) ? a0 + ch : nk;
  double acc   = 0.0;

  if (j < nobs)
    for (int a = a0; a < a1; ++a)
    {
      const double xa = x[a];

      if (xa != 0.0)
        acc = fma (AT[(size_t) a * nobs + j], xa, acc);
    }

  if (j < nobs)
    part[(size_t) blockIdx.y * nobs + j] = acc;
}

__global__ void __launch_bounds__ (256)
k_residual (const double *__restrict__ part, int nch, int nobs, const double *__restrict__ f,
            double *__restrict__ r, double *__restrict__ partial)
{
  __shared__ double red[256];
  const int j = blockIdx.x * 256 + threadIdx.x;
  double rj   = 0.0;

  if (j < nobs)
  {
    double acc = 0.0;

    for (int c = 0; c < nch; ++c)
      acc += part[(size_t) c * nobs + j];

    rj   = (f ? f[j] : 1.0) - acc;
    r[j] = rj;
  }

  red[threadIdx.x] = rj * rj;
  __syncthreads ();

  for (int o = 128; o > 0; o >>= 1)
  {
    if (threadIdx.x < o)
      red[threadIdx.x] += red[threadIdx.x + o];

    __syncthreads ();
  }

  if (threadIdx.x == 0)
    partial[blockIdx.x] = red[0];
}

__global__ void
k_sum_partials (const double *__restrict__ partial, int np, double *__restrict__ out)
{
  if (threadIdx.x == 0 && blockIdx.x == 0)
  {
    double s = 0.0;

    for (int i = 0; i < np; ++i)
      s += partial[i];

    out[0] = s;
  }
}

size_t
residual_work_doubles (int nk, int nobs)
{
  const int ch = res_chunk (nk, nobs);

  return (size_t) ((nk + ch - 1) / ch) * nobs;
}

hipError_t
launch_residual (const double *AT, int nk, int nobs, const double *x, const double *f, double *r, double *partial,
                 double *rnorm2, double *work, hipStream_t s)
{
  const int nb  = (nobs + 255) / 256;
  const int ch  = res_chunk (nk, nobs);
  const int nch = (nk + ch - 1) / ch;

  hipLaunchKernelGGL (k_residual_part, dim3 (nb, nch), dim3 (256), 0, s, AT, nk, nobs, x, ch, work);
  hipLaunchKernelGGL (k_residual, dim3 (nb), dim3 (256), 0, s, work, nch, nobs, f, r, partial);
  hipLaunchKernelGGL (k_sum_partials, dim3 (1), dim3 (64), 0, s, partial, nb, rnorm2);

  return hipGetLastError ();
}

// S = M[P][P], bs = b[P]
__global__ void
k_gather_sym (const double *__restrict__ M, int n, const int *__restrict__ P, int np, double *__restrict__ S,
              const double *__restrict__ b, double *__restrict__ bs)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;

  if (r >= np || c >= np)
    return;

  S[(size_t) r * np + c] = M[(size_t) P[r] * n + P[c]];

  if (c == 0)
    bs[r] = b[P[r]];
}

hipError_t
launch_gather_sym (const double *M, int n, const int *P, int np, double *S, const double *b, double *bs,
                   hipStream_t s)
{
  hipLaunchKernelGGL (k_gather_sym, dim3 ((np + 255) / 256, np), dim3 (256), 0, s, M, n, P, np, S, b, bs);

  return hipGetLastError ();
}

// double broadcast from lane `src` (a compile-time constant after unrolling)
__device__ inline double
bcast_lane (double v, int src)
{
  const int lo = __builtin_amdgcn_readlane (__double2loint (v), src);
  const int hi = __builtin_amdgcn_readlane (__double2hiint (v), src);

  return __hiloint2double (hi, lo);
}

// lower triangle <- transpose of the upper factor (for the backward solve)
__global__ void
k_mirror_lower (double *__restrict__ S, int np)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;

  if (r < np && c < r)
    S[(size_t) r * np + c] = S[(size_t) c * np + r];
}

// S[off:][off:] -= (rank-K product of the rows kb .. kb+K), upper triangle:
// 128-wide tiles while they number at least 16384 (trailing size above
// about 23000: more reuse per staged operand), 64-wide ones below (measured
// faster at n = 20000 and below)
hipError_t
launch_trailing_update (double *S, int np, int K, int off, int kb, hipStream_t s)
{
  const int nt128 = (np - off + 127) / 128;

  if (nt128 * (nt128 + 1) / 2 >= 16384)
    launch_syrk_mfma<128> (S, np, K, np, off, kb, S, s);
  else
    launch_syrk_mfma<64> (S, np, K, np, off, kb, S, s);

  return hipGetLastError ();
}

// U^T y = b then U x = y with the factor of launch_potrf (upper triangle =
// U, lower triangle = U^T), in 64-row panels: one launch per panel and
// direction.  With T[i][j] = S[(p0+j) np + p0+i], the panel's diagonal
// block is L = U^T below its diagonal (forward) and U above it (backward),
// and the coupling of a row i outside the panel to panel column c is
// S[(p0+c) np + i] in both directions, a unit-stride read over i.  Every
// block stages T in LDS and solves the panel with one wave (64 serial
// steps, operands shuffled from the pivot lane); block 0 writes the panel's
// solution to `out`, and every block updates its 256 rows of the right-hand
// side outside the panel.  The panel rows of `rhs` are only read in a
// launch, so the blocks never race.
constexpr int TS_NB = 64;

template <int FWD>
__global__ void __launch_bounds__ (256)
k_trsv_panel (const double *__restrict__ S, int np, int p0, int pb, double *__restrict__ rhs,
              double *__restrict__ out)
{
  __shared__ double T[TS_NB][TS_NB + 1];
  __shared__ double y[TS_NB];
  __shared__ double rdiag[TS_NB];
  const int tid = threadIdx.x;

  {
    double v[16];

#pragma unroll
    for (int q = 0; q < 16; ++q)
    {
      const int e = tid + q * 256, j = e >> 6, i = e & 63;

      v[q] = (i < pb && j < pb) ? S[(size_t) (p0 + j) * np + p0 + i] : 0.0;
    }

#pragma unroll
    for (int q = 0; q < 16; ++q)
    {
      const int e = tid + q * 256;

      T[e & 63][e >> 6] = v[q];
    }
  }

  __syncthreads ();

  if (tid < 64)
  {
    const int i = tid;
    double bi   = (i < pb) ? rhs[p0 + i] : 0.0;

    // reciprocals of the diagonal, then 64 serial steps with the pivot
    // taken by readlane (j is wave-uniform) and a multiplication in place
    // of the division
    rdiag[i] = (i < pb) ? 1.0 / T[i][i] : 0.0;
    __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier ();
    __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");

    if (pb == TS_NB)
    {
      // full panel: the lane's row of T in registers, zero outside the
      // triangle being solved, so each step is a readlane of lane j's
      // scaled value and one fma or select (the same arithmetic as below)
      const double rdl = rdiag[i];
      double t[TS_NB];

#pragma unroll
      for (int j = 0; j < TS_NB; ++j)
        t[j] = (FWD ? (j < i) : (j > i)) ? T[i][j] : 0.0;

#pragma unroll
      for (int step = 0; step < TS_NB; ++step)
      {
        const int j     = FWD ? step : TS_NB - 1 - step;
        const double yj = bcast_lane (bi * rdl, j);

        bi = (i == j) ? yj : fma (-t[j], yj, bi);
      }
    }
    else
    {
      for (int step = 0; step < pb; ++step)
      {
        const int j     = FWD ? step : pb - 1 - step;
        const double bj = bcast_lane (bi, j);
        const double yj = bj * rdiag[j];

        if (i == j)
          bi = yj;
        else if (FWD ? (i > j) : (i < j))
          bi = fma (-T[i][j], yj, bi);
      }
    }

    y[i] = bi;

    if (blockIdx.x == 0 && i < pb)
      out[p0 + i] = bi;
  }

  __syncthreads ();

  const int row = (FWD ? p0 + pb : 0) + blockIdx.x * 256 + tid;
  const int hi  = FWD ? np : p0;

  if (row < hi)
  {
    double t[4] = {rhs[row], 0.0, 0.0, 0.0};

    for (int c0 = 0; c0 < pb; c0 += 16)
    {
      double v[16];

#pragma unroll
      for (int q = 0; q < 16; ++q)
        v[q] = (c0 + q < pb) ? S[(size_t) (p0 + c0 + q) * np + row] : 0.0;

#pragma unroll
      for (int q = 0; q < 16; ++q)
        t[q & 3] = fma (-v[q], (c0 + q < pb) ? y[c0 + q] : 0.0, t[q & 3]);
    }

    rhs[row] = (t[0] + t[1]) + (t[2] + t[3]);
  }
}

// solution of (U^T U) x = b returned in b; tmp holds np doubles
hipError_t
launch_trsv_pair (const double *S, int np, double *b, double *tmp, hipStream_t s)
{
  for (int p0 = 0; p0 < np; p0 += TS_NB)
  {
    const int pb   = (np - p0 < TS_NB) ? np - p0 : TS_NB;
    const int rest = np - p0 - pb;
    const int grid = (rest + 255) / 256 > 0 ? (rest + 255) / 256 : 1;

    hipLaunchKernelGGL (k_trsv_panel<1>, dim3 (grid), dim3 (256), 0, s, S, np, p0, pb, b, tmp);
  }

  const int last = ((np - 1) / TS_NB) * TS_NB;

  for (int p0 = last; p0 >= 0; p0 -= TS_NB)
  {
    const int pb   = (np - p0 < TS_NB) ? np - p0 : TS_NB;
    const int grid = (p0 + 255) / 256 > 0 ? (p0 + 255) / 256 : 1;

    hipLaunchKernelGGL (k_trsv_panel<0>, dim3 (grid), dim3 (256), 0, s, S, np, p0, pb, tmp, b);
  }

  return hipGetLastError ();
}

// U x = y alone, U in the upper triangle and U^T mirrored into the lower one
// (the factor of launch_lu_factor after launch_mirror_lower); y is consumed
hipError_t
launch_trsv_backward (const double *S, int np, double *y, double *x, hipStream_t s)
{
  const int last = ((np - 1) / TS_NB) * TS_NB;

  for (int p0 = last; p0 >= 0; p0 -= TS_NB)
  {
    const int pb   = (np - p0 < TS_NB) ? np - p0 : TS_NB;
    const int grid = (p0 + 255) / 256 > 0 ? (p0 + 255) / 256 : 1;

    hipLaunchKernelGGL (k_trsv_panel<0>, dim3 (grid), dim3 (256), 0, s, S, np, p0, pb, y, x);
  }

  return hipGetLastError ();
}

// The backward sweep as one launch, chained by flags: one 64-lane block per
// panel, block k taking the k-th panel in sweep order (the forward sweep runs
// inside the factorisation, k_potrf.hip).  A block
// applies the contributions of the panels before it in sweep order, each
// as soon as that panel's flag carries this call's epoch, with the order
// and arithmetic of k_trsv_panel (the solution is the same to the bit),
// then solves its diagonal block and publishes its part of the solution and
// its flag.  The factor entries of a contribution are loaded before its
// flag is awaited.  The host launches the chain only when every block of
// the grid can be resident at once, so each wait ends; a wait longer than
// spin_limit polls still ends the kernel, with *status = epoch (no later
// block does anything then), and the host solves again with
// the panel launches.
__global__ void __launch_bounds__ (64)
k_trsv_chain (const double *__restrict__ S, int np, const double *__restrict__ rhs, double *__restrict__ out,
              unsigned *__restrict__ flags, unsigned epoch, unsigned spin_limit, unsigned *__restrict__ status)
{
  __shared__ double T[TS_NB][TS_NB + 1];
  __shared__ double rdiag[TS_NB];
  __shared__ double ys[TS_NB];
  const int lane = threadIdx.x;
  const int npan = (np + TS_NB - 1) / TS_NB;
  const int k    = blockIdx.x;
  const int pan  = npan - 1 - k;
  const int p0   = pan * TS_NB;
  const int pb   = (np - p0 < TS_NB) ? np - p0 : TS_NB;

  if (__hip_atomic_load (status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch)
    return;

  for (int e = lane; e < TS_NB * TS_NB; e += 64)
  {
    const int j = e >> 6, i = e & 63;

    T[i][j] = (i < pb && j < pb) ? S[(size_t) (p0 + j) * np + p0 + i] : 0.0;
  }

  const int row = p0 + lane;
  double r      = (lane < pb) ? rhs[row] : 0.0;

  for (int kk = 0; kk < k; ++kk)
  {
    const int q  = npan - 1 - kk;
    const int q0 = q * TS_NB;
    const int qb = (np - q0 < TS_NB) ? np - q0 : TS_NB;
    double v[TS_NB];

#pragma unroll
    for (int c = 0; c < TS_NB; ++c)
      v[c] = (c < qb && lane < pb) ? S[(size_t) (q0 + c) * np + row] : 0.0;

    unsigned polls = 0;
    bool dead      = false;

    while (__hip_atomic_load (&flags[q], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) != epoch)
    {
      if (++polls > spin_limit || __hip_atomic_load (status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch)
      {
        dead = true;
        break;
      }

      __builtin_amdgcn_s_sleep (1);
    }

    if (dead)
    {
      if (lane == 0)
        __hip_atomic_store (status, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

      return;
    }

    ys[lane] = (lane < qb) ? out[q0 + lane] : 0.0;
    __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier ();
    __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");

    double t[4] = {r, 0.0, 0.0, 0.0};

#pragma unroll
    for (int c0 = 0; c0 < TS_NB; c0 += 16)
#pragma unroll
      for (int qq = 0; qq < 16; ++qq)
        if (c0 < qb)
          t[qq & 3] = fma (-v[c0 + qq], (c0 + qq < qb) ? ys[c0 + qq] : 0.0, t[qq & 3]);

    r = (t[0] + t[1]) + (t[2] + t[3]);
    __builtin_amdgcn_wave_barrier ();
  }

  __syncthreads ();

  const int i = lane;
  double bi   = r;

  rdiag[i] = (i < pb) ? 1.0 / T[i][i] : 0.0;
  __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier ();
  __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");

  if (pb == TS_NB)
  {
    const double rdl = rdiag[i];
    double t[TS_NB];

#pragma unroll
    for (int j = 0; j < TS_NB; ++j)
      t[j] = (j > i) ? T[i][j] : 0.0;

#pragma unroll
    for (int step = 0; step < TS_NB; ++step)
    {
      const int j     = TS_NB - 1 - step;
      const double yj = bcast_lane (bi * rdl, j);

      bi = (i == j) ? yj : fma (-t[j], yj, bi);
    }
  }
  else
  {
    for (int step = 0; step < pb; ++step)
    {
      const int j     = pb - 1 - step;
      const double bj = bcast_lane (bi, j);
      const double yj = bj * rdiag[j];

      if (i == j)
        bi = yj;
      else if (i < j)
        bi = fma (-T[i][j], yj, bi);
    }
  }

  if (i < pb)
    out[p0 + i] = bi;

  __hip_atomic_store (&flags[pan], epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// panels the chained sweeps take at most: the blocks of k_trsv_chain the
// device holds at once
int
trsv_chain_max_panels ()
{
  static const int cap = [] {
    int dev = 0, ncu = 0, nb = 0;

    (void) hipGetDevice (&dev);
    (void) hipDeviceGetAttribute (&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    (void) hipOccupancyMaxActiveBlocksPerMultiprocessor (&nb, k_trsv_chain, 64, 0);
    return (nb > 0 && ncu > 0) ? nb * ncu : 0;
  }();

  return cap;
}

// flags: status word, then npan panel flags
hipError_t
launch_trsv_chain (const double *S, int np, const double *y, double *x, unsigned *flags, unsigned epoch, hipStream_t s)
{
  const int npan = (np + TS_NB - 1) / TS_NB;

  hipLaunchKernelGGL (k_trsv_chain, dim3 (npan), dim3 (64), 0, s, S, np, y, x, flags + 1, epoch, 1u << 22, flags);

  return hipGetLastError ();
}

hipError_t
launch_mirror_lower (double *S, int np, hipStream_t s)
{
  hipLaunchKernelGGL (k_mirror_lower, dim3 ((np + 255) / 256, np), dim3 (256), 0, s, S, np);

  return hipGetLastError ();
}

__global__ void
k_scatter (const double *__restrict__ sol, const int *__restrict__ P, int np, int n, double *__restrict__ x)
{
  const int a = blockIdx.x * blockDim.x + threadIdx.x;

  if (a < n)
    x[a] = 0.0;
}

__global__ void
k_scatter2 (const double *__restrict__ sol, const int *__restrict__ P, int np, double *__restrict__ x)
{
  const int a = blockIdx.x * blockDim.x + threadIdx.x;

  if (a < np)
    x[P[a]] = sol[a];
}

hipError_t
launch_scatter (const double *sol, const int *P, int np, int n, double *x, hipStream_t s)
{
  hipLaunchKernelGGL (k_scatter, dim3 ((n + 255) / 256), dim3 (256), 0, s, sol, P, np, n, x);
  hipLaunchKernelGGL (k_scatter2, dim3 ((np + 255) / 256), dim3 (256), 0, s, sol, P, np, x);

  return hipGetLastError ();
}

// w <- w (1 - s) / sum(w) + s / n  (ncm_stats_dist.c:1087-1093), serial sum
__global__ void
k_shrink (double *__restrict__ w, int n, double shrink, int *__restrict__ status)
{
  __shared__ double total;
  __shared__ double wl[4096];
  double t = 0.0;

  // serial sum in index order (thread 0) over chunks staged in LDS
  for (int i0 = 0; i0 < n; i0 += 4096)
  {
    const int cnt = (n - i0 < 4096) ? n - i0 : 4096;

    for (int i = threadIdx.x; i < cnt; i += blockDim.x)
      wl[i] = w[i0 + i];

    __syncthreads ();

    if (threadIdx.x == 0)
      for (int i = 0; i < cnt; ++i)
        t = __dadd_rn (t, wl[i]);

    __syncthreads ();
  }

  if (threadIdx.x == 0)
  {
    total = t;

    if (!(t > 0.0))
      status[0] = 3;
  }

  __syncthreads ();

  const double sc = (1.0 - shrink) / total;
  const double ad = shrink / n;

  for (int i = threadIdx.x; i < n; i += blockDim.x)
    w[i] = __dadd_rn (__dmul_rn (w[i], sc), ad);
}

hipError_t
launch_shrink (double *w, int n, double shrink, int *status, hipStream_t s)
{
  hipLaunchKernelGGL (k_shrink, dim3 (1), dim3 (1024), 0, s, w, n, shrink, status);

  return hipGetLastError ();
}

} // namespace nck

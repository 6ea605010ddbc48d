// kde_tile.h -- |W_i (x - theta_i)|^2 of 64 pairs per wave on the matrix
// cores, shared by the FP64 / FP32 evaluations and the interpolation matrix
// of the VKDE from 13 dimensions on.
//
// z = W_i delta, delta = x - theta_i (formed in FP64 per pair, as the vector
// form does), on 16 x 16 x 4 MFMA tiles: A = 16 rows of W_i by 4 columns,
// B = 4 coordinates of delta by 16 points.  A wave holds NT point tiles; a
// fragment of W_i, gathered from the packed lower triangle, feeds all of
// them.  Of the 4 NK columns (NK = ceil (d / 4)), row tile rt takes the
// K steps up to its diagonal block only, entries above the diagonal are
// masked, and the K loop is the outer one, so that delta lives for one step.
//
// Why not the vector units: there every entry of W_i is an SGPR operand, and
// the scalar cache delivers about 8 B per cycle: at d = 16 a kernel's 1.2 KB
// take twice as long as its 136 FMAs, and the 16.6 KB of d = 64 (more than
// the whole scalar cache) eight times.  On the matrix cores an entry is read
// once per 16 x NT points through the vector L1.  The triangle costs
// 16 NRT (NRT + 1) / 2 instead of D (D + 1) / 2 rows-by-columns / D, 1.9x
// the FMAs at d = 16 and 1.2x at d = 64; up to d = 12 the vector form wins.
#pragma once

#include <hip/hip_runtime.h>

namespace nck
{

typedef double tile_f64x4 __attribute__ ((ext_vector_type (4)));
typedef float tile_f32x4 __attribute__ ((ext_vector_type (4)));

template <typename T> struct TileAcc;
template <> struct TileAcc<double> { typedef tile_f64x4 V; };
template <> struct TileAcc<float> { typedef tile_f32x4 V; };

__device__ inline tile_f64x4
tile_mfma (double a, double b, tile_f64x4 c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64 (a, b, c, 0, 0, 0);
}

__device__ inline tile_f32x4
tile_mfma (float a, float b, tile_f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32 (a, b, c, 0, 0, 0);
}

// a + b exchanged across the halves of the wave: lanes 0-31 get a[l] +
// a[l + 32], lanes 32-63 get b[l] + b[l - 32]
__device__ inline float
tile_swap32 (float a, float b)
{
  const auto r = __builtin_amdgcn_permlane32_swap (__float_as_uint (a), __float_as_uint (b), false, false);

  return __uint_as_float (r[0]) + __uint_as_float (r[1]);
}

__device__ inline double
tile_swap32 (double a, double b)
{
  const auto lo = __builtin_amdgcn_permlane32_swap ((unsigned) __double2loint (a), (unsigned) __double2loint (b),
                                                    false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap ((unsigned) __double2hiint (a), (unsigned) __double2hiint (b),
                                                    false, false);

  return __hiloint2double ((int) hi[0], (int) lo[0]) + __hiloint2double ((int) hi[1], (int) lo[1]);
}

// the same across the 16-lane rows: even rows get a of both rows of their
// pair, odd rows b
__device__ inline float
tile_swap16 (float a, float b)
{
  const auto r = __builtin_amdgcn_permlane16_swap (__float_as_uint (a), __float_as_uint (b), false, false);

  return __uint_as_float (r[0]) + __uint_as_float (r[1]);
}

__device__ inline double
tile_swap16 (double a, double b)
{
  const auto lo = __builtin_amdgcn_permlane16_swap ((unsigned) __double2loint (a), (unsigned) __double2loint (b),
                                                    false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap ((unsigned) __double2hiint (a), (unsigned) __double2hiint (b),
                                                    false, false);

  return __hiloint2double ((int) hi[0], (int) lo[0]) + __hiloint2double ((int) hi[1], (int) lo[1]);
}

// Point tiles per wave: the coordinates take 2 NT NK registers and the FP64
// accumulators 8 NT NRT, so 4 tiles up to d = 32 and 2 above (two waves per
// SIMD either way).  With 2 tiles a step takes 2 kernels, so that all 64
// lanes hold a pair in the terms.  FP32 accumulators take half of that, and
// an FP32 step half the time of an FP64 one while its fragments of W_i cost the
// vector L1 the same 16 lines: 4 tiles always (FP32, n = 8000, m = 40000: 28.4
// against 16.8 ms at d = 64, 15.1 against 8.9-11.7 at d = 40).
template <typename T>
constexpr int
tile_nt (int NK)
{
  return (NK <= 8 || sizeof (T) == 4) ? 4 : 2;
}

template <typename T, int NK>
struct PairTile
{
  static constexpr int NT  = tile_nt<T> (NK);
  static constexpr int KU  = 4 / NT;            // kernels per step
  static constexpr int NRT = (NK + 3) / 4;      // row tiles
  static constexpr int PTS = 16 * NT;           // points per wave
  typedef typename TileAcc<T>::V V;

  double x[NT][NK];    // coordinate 4 s + lane / 16 of point 16 t + lane % 16
  int ro[NRT];         // packed offset of row 16 rt + lane % 16, plus lane / 16
  int li, lk, D;

  // point p0 + q of the wave, clamped to the last of the m points
  __device__ inline void
  load_points (const double *__restrict__ X, int p0, int m, int d, int D_)
  {
    const int lane = threadIdx.x & 63;

    li = lane & 15;
    lk = lane >> 4;
    D  = D_;

#pragma unroll
    for (int t = 0; t < NT; ++t)
    {
      const int p       = min (p0 + 16 * t + li, m - 1);
      const double *row = X + (size_t) p * d;

#pragma unroll
      for (int s = 0; s < NK; ++s)
        x[t][s] = (4 * s + lk < d) ? row[4 * s + lk] : 0.0;
    }

#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
    {
      const int r = min (16 * rt + li, D - 1);   // rows past D are masked

      ro[rt] = r * (r + 1) / 2 + lk;
    }
  }

  // the pair of a lane: point (in the wave) and kernel (in the step)
  __device__ inline int
  lane_point () const
  {
    const int lane = threadIdx.x & 63;

    return (NT == 4) ? lane : (lane >> 5) * 16 + (lane & 15);
  }

  __device__ inline int
  lane_kernel () const
  {
    return (NT == 4) ? 0 : ((threadIdx.x >> 4) & 1);
  }

  // partial squared norms of kernel i (this lane's rows of every tile)
  template <typename WT>
  __device__ inline void
  partials (const WT *__restrict__ Wp, const double *__restrict__ Th, int i, T (&part)[NT]) const
  {
    const WT *W      = Wp + (size_t) i * (D * (D + 1) / 2);   // wave-uniform base
    const double *th = Th + (size_t) i * D;
    V acc[NRT][NT];

#pragma unroll
    for (int s = 0; s < NK; ++s)
    {
      const double c = th[4 * s + lk];
      T delta[NT];

#pragma unroll
      for (int t = 0; t < NT; ++t)
        delta[t] = (T) (x[t][s] - c);

#pragma unroll
      for (int rt = s / 4; rt < NRT; ++rt)
      {
        T a = (T) W[ro[rt] + 4 * s];

        // the diagonal block keeps columns up to the row; rows past D are zero
        if (s / 4 == rt && 4 * (s - 4 * rt) + lk > li)
          a = (T) 0;

        if (rt == NRT - 1 && 16 * NRT > 4 * NK && 16 * rt + li >= D)
          a = (T) 0;

#pragma unroll
        for (int t = 0; t < NT; ++t)
        {
          const V zero = {(T) 0, (T) 0, (T) 0, (T) 0};

          acc[rt][t] = tile_mfma (a, delta[t], (s == 0) ? zero : acc[rt][t]);
        }
      }
    }

#pragma unroll
    for (int t = 0; t < NT; ++t)
    {
      T p = (T) 0;

#pragma unroll
      for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p = fma (acc[rt][t][r], acc[rt][t][r], p);

      part[t] = p;
    }
  }

  // squared norm of the lane's pair: kernel i + lane_kernel () (the last one
  // is repeated past i1) and point lane_point ()
  template <typename WT>
  __device__ inline T
  chi2 (const WT *__restrict__ Wp, const double *__restrict__ Th, int i, int i1) const
  {
    if constexpr (NT == 4)
    {
      T p[NT];

      partials (Wp, Th, i, p);

      return tile_swap16 (tile_swap32 (p[0], p[2]), tile_swap32 (p[1], p[3]));
    }
    else
    {
      T p[NT], q[NT];

      partials (Wp, Th, i, p);
      partials (Wp, Th, min (i + 1, i1 - 1), q);

      return tile_swap16 (tile_swap32 (p[0], p[1]), tile_swap32 (q[0], q[1]));
    }
  }
};

// NK of the instantiations: the next at or above ceil (d / 4)
inline int
tile_nk (int d)
{
  const int nk = (d + 3) / 4;

  return (nk <= 8) ? nk : ((nk + 1) & ~1);
}

} // namespace nck

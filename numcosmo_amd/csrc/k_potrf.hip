// k_potrf.hip -- blocked Cholesky of the normal equations, with the forward
// substitution of their right-hand side.
//
// S = U^T U (upper, as dposv with the row-major 'U' of ncm_matrix.c:1198-1208)
// in 64-row panels, right-looking, one launch per panel.  What bounds it is
// the serial chain of panels: a panel's update by the one before it, its 64
// pivot steps, and a launch.  A launch therefore holds everything that does
// not wait for its own panel:
//   panel blocks (first in the grid): each updates its 64 x 64 tile of panel
//     k's rows and, redundantly, the diagonal block by panel k - 1 on the FP64
//     matrix cores, then factors the diagonal block and solves its 64 columns;
//   tile blocks: the update of the rows below panel k by panel k - 1;
//   right-hand-side blocks: b below panel k minus U_{k-1}^T y_{k-1}.
// The tiles thus run beside the next panel's pivots instead of before them.
// n = 3200, factor and forward sweep: 2.28 ms with separate panel and update
// launches (27 + 13 us per panel) and a sweep of its own, 1.31 ms (26 us per
// panel: update 8, pivots 8, solves of the other columns 4) here.
#include "kde_math.h"
#include "nckde_internal.h"

namespace nck
{

typedef double f64x4 __attribute__ ((ext_vector_type (4)));

constexpr int CH_NB  = 64;
constexpr int CH_LD  = CH_NB + 4;   // LDS row stride
constexpr int SP_NB  = 4 * CH_NB;   // super-panel: four panels
constexpr int SP_MIN = 4096;        // columns left above which super-panels are used

struct StepArgs
{
  double *S;
  int np, kb, upd;       // upd: rows from kb on still lack the update by panel kb - 64
  int *info;             // first failing pivot + 1 (LAPACK), else 0
  double *Ud;            // factored diagonal block (row-major 64 x 64, upper)
  double *b;             // right-hand side: y = U^{-T} b in place
  int npb, nrb, ntiles;
};

// double broadcast from lane `src` (wave-uniform)
__device__ inline double
lane_bcast (double v, int src)
{
  const int lo = __builtin_amdgcn_readlane (__double2loint (v), src);
  const int hi = __builtin_amdgcn_readlane (__double2hiint (v), src);

  return __hiloint2double (hi, lo);
}

// Entry (w + 4 q, lane) of the 64 x 64 tile at (r0, c0) in v[q], `eye` or 0 past
// np.  The row is wave-uniform, so that its address is scalar work; rows and
// columns out of range read element 0.
__device__ inline void
load_tile (const double *__restrict__ S, int np, int r0, int c0, bool eye, double (&v)[16])
{
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const bool cin = c0 + lane < np;
  const int col  = cin ? c0 + lane : 0;

#pragma unroll
  for (int q = 0; q < 16; ++q)
  {
    const int r      = w + 4 * q;
    const bool in    = r0 + r < np;
    const double *at = S + (in ? (size_t) (r0 + r) * np : 0);
    const double t   = at[col];

    v[q] = (in && cin) ? t : ((eye && r == lane) ? 1.0 : 0.0);
  }
}

__device__ inline void
store_tile (double (&T)[CH_NB][CH_LD], const double (&v)[16])
{
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;

#pragma unroll
  for (int q = 0; q < 16; ++q)
    T[w + 4 * q][lane] = v[q];
}

// acc -= A^T B over the 64 staged rows for the 32 x 32 quarter (wr, wc)
__device__ inline void
quarter_product (const double (&A)[CH_NB][CH_LD], const double (&B)[CH_NB][CH_LD], int wr, int wc, f64x4 (&acc)[2][2])
{
  const int li = threadIdx.x & 15, lk = (threadIdx.x >> 4) & 3;

#pragma unroll
  for (int ks = 0; ks < CH_NB / 4; ++ks)
  {
    const int kq = 4 * ks + lk;
    double fa[2], fb[2];

#pragma unroll
    for (int i = 0; i < 2; ++i)
    {
      fa[i] = -A[kq][wr + 16 * i + li];
      fb[i] = B[kq][wc + 16 * i + li];
    }

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64 (fa[i], fb[j], acc[i][j], 0, 0, 0);
  }
}

// One 64 x 64 tile of the trailing update.  All loads (both panels' rows and
// the tile itself) are in flight before the first wait.
__device__ inline void
update_tile (const StepArgs &a, int r0, int c0, double (&As)[CH_NB][CH_LD], double (&Bs)[CH_NB][CH_LD])
{
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr   = (w >> 1) * 32, wc = (w & 1) * 32;
  const int li   = lane & 15, lk = lane >> 4;
  const bool all = (r0 + CH_NB <= a.np && c0 + CH_NB <= a.np && c0 > r0);
  f64x4 acc[2][2];
  double va[16], vb[16];
  double *tp = a.S + (size_t) (r0 + wr + lk) * a.np + c0 + wc + li;   // element (0, 0, 0) of this lane

  auto in = [&] (int i, int j, int r) {
    const int row = r0 + wr + 16 * i + lk + 4 * r, col = c0 + wc + 16 * j + li;

    return all || (row < a.np && col < a.np && row <= col);
  };

  load_tile (a.S, a.np, a.kb - CH_NB, r0, false, va);
  load_tile (a.S, a.np, a.kb - CH_NB, c0, false, vb);

#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < 2; ++j)
      {
        const double *at = in (i, j, r) ? tp + (size_t) (16 * i + 4 * r) * a.np + 16 * j : a.S;

        acc[i][j][r] = *at;
      }

  store_tile (As, va);
  store_tile (Bs, vb);
  __syncthreads ();
  quarter_product (As, Bs, wr, wc, acc);

#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (in (i, j, r))
          tp[(size_t) (16 * i + 4 * r) * a.np + 16 * j] = acc[i][j][r];
}

// a pivot failed in an earlier panel (a failure of this launch is above kb
// and does not count, so that every wave of a block decides alike)
__device__ inline bool
pivot_failed (const StepArgs &a)
{
  const int failed = *a.info;

  return failed != 0 && failed <= a.kb;
}

constexpr int CH_SB = 16;   // rows of a sub-panel

// Rows 16 sb .. 16 sb + 15 of the factor for the 64 columns of the diagonal
// block, one per lane, by one wave.  The next pivot's row goes first, with a
// readlane factor, so that its chain (two readlanes, an inverse root, a
// product) runs under the update of the others, whose factors are read back
// from the published row (a readlane pair per factor took twice the cycles).
// Entries below the diagonal take part unmasked: they only combine with each
// other.  Returns the first non-positive pivot + 1 within the panel, else 0: its
// diagonal entry, and no earlier one, is NaN (an inverse root of a value
// not above zero, times that value).
__device__ inline int
pivot_rows (double (&Ds)[CH_NB][CH_LD], double (&Rr)[CH_NB], int sb, int lane)
{
  const int r0 = CH_SB * sb;
  double x[CH_SB];
  double ujj = 1.0, rj = 0.0;   // lane j: its row's pivot root and inverse

#pragma unroll
  for (int i = 0; i < CH_SB; ++i)
    x[i] = Ds[r0 + i][lane];

  double rn = rsqrt_f64 (lane_bcast (x[0], r0));

#pragma unroll
  for (int j = 0; j < CH_SB; ++j)
  {
    double dn = 1.0, re = 1.0;

    x[j] = x[j] * rn;
    ujj  = (lane == r0 + j) ? x[j] : ujj;
    rj   = (lane == j) ? rn : rj;

    Ds[r0 + j][lane] = x[j];

    if (j + 1 < CH_SB)
    {
      x[(j + 1) % CH_SB] = fma (-lane_bcast (x[j], r0 + j + 1), x[j], x[(j + 1) % CH_SB]);
      dn                 = lane_bcast (x[(j + 1) % CH_SB], r0 + j + 1);
      re                 = __builtin_amdgcn_rsq (dn);
    }

    // the rows from j + 2 on, factors from the row just published
    __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier ();
    __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");
    rn = rsqrt_step (dn, re);

#pragma unroll
    for (int i = j + 2; i < CH_SB; ++i)
      x[i] = fma (-Ds[r0 + j][r0 + i], x[j], x[i]);
  }

  if (lane < CH_SB)
    Rr[r0 + lane] = rj;

  const unsigned long long bad = __ballot (!(ujj > 0.0));

  return bad ? (int) __ffsll (bad) : 0;
}

// the same rows of 64 other columns (column col of a lane), after pivot_rows
__device__ inline void
follow_rows (const double (&Ds)[CH_NB][CH_LD], const double (&Rr)[CH_NB], double (&Os)[CH_NB][CH_LD], int sb, int col,
             bool store)
{
  const int r0 = CH_SB * sb;
  double x[CH_SB];

#pragma unroll
  for (int i = 0; i < CH_SB; ++i)
    x[i] = Os[r0 + i][col];

#pragma unroll
  for (int j = 0; j < CH_SB; ++j)
  {
    x[j] = x[j] * Rr[r0 + j];

#pragma unroll
    for (int i = j + 1; i < CH_SB; ++i)
      x[i] = fma (-Ds[r0 + j][r0 + i], x[j], x[i]);
  }

  if (store)
  {
#pragma unroll
    for (int i = 0; i < CH_SB; ++i)
      Os[r0 + i][col] = x[i];
  }
}

// 16 x 16 blocks minus the product of sub-panel sb's rows (columns 16 ti of
// the diagonal block by columns 16 tj of the block's tile), two at a time:
// their LDS reads and MFMA chains overlap.  Blocks are numbered row by row:
// the own tile's rows t0 .. 3 (4 columns each), then the diagonal block's
// upper rows d0 .. 3.
struct SubBlock
{
  int own, ti, tj;
};

__device__ inline SubBlock
sub_block (int t, int t0, int n_own, int d0)
{
  if (t < n_own)
    return {1, t0 + t / 4, t % 4};

  int ti = d0;

  t -= n_own;

  while (t >= 4 - ti)
  {
    t -= 4 - ti;
    ++ti;
  }

  return {0, ti, ti + t};
}

__device__ inline void
sub_update2 (double (&Ls)[2][CH_NB][CH_LD], int sb, SubBlock p, SubBlock q, bool two, int lane)
{
  const int li = lane & 15, lk = lane >> 4;
  f64x4 a, b;
  double pa[4], pb[4], qa[4], qb[4];

#pragma unroll
  for (int r = 0; r < 4; ++r)
  {
    const int k = CH_SB * sb + 4 * r + lk;

    a[r]  = Ls[p.own][16 * p.ti + lk + 4 * r][16 * p.tj + li];
    b[r]  = Ls[q.own][16 * q.ti + lk + 4 * r][16 * q.tj + li];
    pa[r] = -Ls[0][k][16 * p.ti + li];
    qa[r] = -Ls[0][k][16 * q.ti + li];
    pb[r] = Ls[p.own][k][16 * p.tj + li];
    qb[r] = Ls[q.own][k][16 * q.tj + li];
  }

#pragma unroll
  for (int r = 0; r < 4; ++r)
  {
    a = __builtin_amdgcn_mfma_f64_16x16x4f64 (pa[r], pb[r], a, 0, 0, 0);
    b = __builtin_amdgcn_mfma_f64_16x16x4f64 (qa[r], qb[r], b, 0, 0, 0);
  }

#pragma unroll
  for (int r = 0; r < 4; ++r)
  {
    Ls[p.own][16 * p.ti + lk + 4 * r][16 * p.tj + li] = a[r];

    if (two)
      Ls[q.own][16 * q.ti + lk + 4 * r][16 * q.tj + li] = b[r];
  }
}

// blocks first, first + step, ... below n
__device__ inline void
sub_updates (double (&Ls)[2][CH_NB][CH_LD], int sb, int first, int step, int n, int t0, int n_own, int d0, int lane)
{
  for (int t = first; t < n; t += 2 * step)
  {
    const bool two = t + step < n;

    sub_update2 (Ls, sb, sub_block (t, t0, n_own, d0), sub_block (two ? t + step : t, t0, n_own, d0), two, lane);
  }
}

// Panel kb for the 64 columns from c0, in four sub-panels of 16 rows.  Wave 0
// runs the pivots, 16 at a time; wave 1 then solves the block's own columns
// for these rows (wave 2 of block 0 the right-hand side, held as column 64 of
// the own tile) while waves 0, 2 and 3 update the next 16 rows of the diagonal
// block; what is below them runs beside the next 16 pivots.  The whole panel
// unrolled over its 64 steps was bound by the instruction fetch of 60 KB of
// straight-line code (42 us); sub-panels are loops over 4 KB (17 us).  Columns past np
// are those of the identity.  A non-positive pivot is recorded (the first
// one), the steps run on, and what they store is not used.
__device__ inline void
panel_block (const StepArgs &a, double (&Ls)[2][CH_NB][CH_LD])
{
  double (&As)[CH_NB][CH_LD] = Ls[0];
  double (&Bs)[CH_NB][CH_LD] = Ls[1];
  __shared__ double Rr[CH_NB];
  __shared__ int s_fail;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li   = lane & 15, lk = lane >> 4;
  const int c0   = a.kb + CH_NB + blockIdx.x * CH_NB;
  const bool own = c0 < a.np;

  // right-hand side (block 0): b of the panel's rows and y of the one before
  const bool rhs = (blockIdx.x == 0 && w == 2);
  double bl = 0.0, yl = 0.0;

  if (rhs)
  {
    bl = (a.kb + lane < a.np) ? a.b[a.kb + lane] : 0.0;
    yl = (a.kb > 0) ? a.b[a.kb - CH_NB + lane] : 0.0;
  }

  // the rows the panel's product needs (or, without one, the panel itself)
  double va[16], vb[16];
  const int src = a.upd ? a.kb - CH_NB : a.kb;

  load_tile (a.S, a.np, src, a.kb, !a.upd, va);

  if (own)
    load_tile (a.S, a.np, src, c0, false, vb);

  if (a.upd)
  {
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
    f64x4 acc[2][2], dacc[3];

    // the diagonal block's 10 upper 16 x 16 blocks, dealt over the waves
    const int e1  = w + 4, e2 = (w + 8 < 10) ? w + 8 : 9;
    const int di1 = (e1 < 7) ? 1 : 2, dj1 = (e1 < 7) ? e1 - 3 : e1 - 5;
    const int di2 = (e2 < 9) ? 2 : 3, dj2 = 3;

    // the products start from the entries themselves, in the MFMA layout
    auto diag_in = [&] (int ti, int tj, int r) {
      const int row = 16 * ti + lk + 4 * r, col = 16 * tj + li;
      const bool in = (a.kb + row < a.np && a.kb + col < a.np);
      const double v = a.S[in ? (size_t) (a.kb + row) * a.np + a.kb + col : 0];

      return in ? v : ((row == col) ? 1.0 : 0.0);
    };

#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
      dacc[0][r] = diag_in (0, w, r);
      dacc[1][r] = diag_in (di1, dj1, r);
      dacc[2][r] = diag_in (di2, dj2, r);
    }

    const double *tp = a.S + (size_t) (a.kb + wr + lk) * a.np;

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
          const int col = c0 + wc + 16 * j + li;

          acc[i][j][r] = *((col < a.np) ? tp + (size_t) (16 * i + 4 * r) * a.np + col : a.S);
        }

    if (pivot_failed (a))
      return;

    store_tile (As, va);

    if (own)
      store_tile (Bs, vb);

    __syncthreads ();

    if (own)
      quarter_product (As, Bs, wr, wc, acc);

    // b minus U_{k-1}^T y_{k-1}, from the staged rows
    if (rhs)
    {
      double t[4] = {bl, 0.0, 0.0, 0.0};

#pragma unroll 8
      for (int k = 0; k < CH_NB; ++k)
        t[k & 3] = fma (-As[k][lane], lane_bcast (yl, k), t[k & 3]);

      bl = (t[0] + t[1]) + (t[2] + t[3]);
    }

#pragma unroll 4
    for (int ks = 0; ks < CH_NB / 4; ++ks)
    {
      const double *row = As[4 * ks + lk];

      dacc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64 (-row[li], row[16 * w + li], dacc[0], 0, 0, 0);
      dacc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64 (-row[16 * di1 + li], row[16 * dj1 + li], dacc[1], 0, 0, 0);

      if (w < 2)
        dacc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64 (-row[16 * di2 + li], row[16 * dj2 + li], dacc[2], 0, 0, 0);
    }

    __syncthreads ();

#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
      As[lk + 4 * r][16 * w + li]               = dacc[0][r];
      As[16 * di1 + lk + 4 * r][16 * dj1 + li]  = dacc[1][r];

      if (w < 2)
        As[16 * di2 + lk + 4 * r][16 * dj2 + li] = dacc[2][r];
    }

    if (own)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Bs[wr + 16 * i + lk + 4 * r][wc + 16 * j + li] = acc[i][j][r];
  }
  else
  {
    if (pivot_failed (a))
      return;

    store_tile (As, va);

    if (own)
      store_tile (Bs, vb);

    // the first panel after a super-panel: b still lacks the last one's part
    if (rhs && a.kb > 0)
    {
      double t[4] = {bl, 0.0, 0.0, 0.0}, v[16];
      const int col = (a.kb + lane < a.np) ? a.kb + lane : a.np - 1;

      for (int k0 = 0; k0 < CH_NB; k0 += 16)
      {
#pragma unroll
        for (int k = 0; k < 16; ++k)
          v[k] = a.S[(size_t) (a.kb - CH_NB + k0 + k) * a.np + col];

#pragma unroll
        for (int k = 0; k < 16; ++k)
          t[k & 3] = fma (-v[k], lane_bcast (yl, k0 + k), t[k & 3]);
      }

      bl = (t[0] + t[1]) + (t[2] + t[3]);
    }
  }

  if (rhs)
    Bs[lane][CH_NB] = bl;   // column 64 of the own tile

  __syncthreads ();

  int fail = 0;

  for (int sb = 0; sb < CH_NB / CH_SB; ++sb)
  {
    if (w == 0)
    {
      const int f = pivot_rows (As, Rr, sb, lane);

      fail = (fail == 0) ? f : fail;
    }
    else if (sb > 0)
    {
      // what sub-panel sb - 1 leaves: the right-hand side and the own tile
      // from row 16 sb on, the diagonal block from row 16 (sb + 1) on
      if (rhs)
      {
        double t[4] = {Bs[lane][CH_NB], 0.0, 0.0, 0.0};

#pragma unroll
        for (int k = CH_SB * (sb - 1), q = 0; q < CH_SB; ++q)
          t[q & 3] = fma (-As[k + q][lane], Bs[k + q][CH_NB], t[q & 3]);

        if (lane >= CH_SB * sb)
          Bs[lane][CH_NB] = (t[0] + t[1]) + (t[2] + t[3]);
      }

      const int n_own = own ? 4 * (4 - sb) : 0;

      sub_updates (Ls, sb - 1, w - 1, 3, n_own + (3 - sb) * (4 - sb) / 2, sb, n_own, sb + 1, lane);
    }

    __syncthreads ();

    if (w == 1)
    {
      if (own)
        follow_rows (As, Rr, Bs, sb, lane, true);
    }
    else
    {
      if (rhs)
        follow_rows (As, Rr, Bs, sb, CH_NB, lane == 0);

      // the next 16 rows of the diagonal block (wave 2 has the right-hand side)
      if (w != 2)
        sub_updates (Ls, sb, (w == 0) ? 0 : 1, 2, 3 - sb, 0, 0, sb + 1, lane);
    }

    __syncthreads ();
  }

  if (threadIdx.x == 0)
    s_fail = fail;

  __syncthreads ();

  if (s_fail != 0)
  {
    if (blockIdx.x == 0 && threadIdx.x == 0)
      *a.info = a.kb + s_fail;

    return;
  }

  if (blockIdx.x == 0)
  {
    for (int r = w; r < CH_NB; r += 4)
      a.Ud[r * CH_NB + lane] = As[r][lane];   // upper part; the rest is never read

    if (w == 0 && a.kb + lane < a.np)
      a.b[a.kb + lane] = Bs[lane][CH_NB];
  }

  if (c0 + lane < a.np)
    for (int r = w; r < CH_NB; r += 4)
      a.S[(size_t) (a.kb + r) * a.np + c0 + lane] = Bs[r][lane];
}

__global__ void __launch_bounds__ (256, 2)
k_potrf_step (StepArgs a)
{
  __shared__ double Ls[2][CH_NB][CH_LD];
  const int bid = blockIdx.x;

  if (bid < a.npb)
  {
    panel_block (a, Ls);
    return;
  }

  if (pivot_failed (a))
    return;

  if (bid < a.npb + a.nrb)
  {
    const int row = a.kb + CH_NB + (bid - a.npb) * 256 + threadIdx.x;

    if (row >= a.np)
      return;

    double t[4] = {a.b[row], 0.0, 0.0, 0.0};

#pragma unroll 16
    for (int k = 0; k < CH_NB; ++k)
      t[k & 3] = fma (-a.S[(size_t) (a.kb - CH_NB + k) * a.np + row], a.b[a.kb - CH_NB + k], t[k & 3]);

    a.b[row] = (t[0] + t[1]) + (t[2] + t[3]);
    return;
  }

  // tiles in contiguous bands per XCD (blocks are dealt round-robin)
  const int per = (gridDim.x - a.npb - a.nrb) / 8;
  const int q   = bid - a.npb - a.nrb;
  int t         = (q % 8) * per + q / 8;

  if (t >= a.ntiles)
    return;

  const int off = a.kb + CH_NB;
  const int nt  = (a.np - off + CH_NB - 1) / CH_NB;
  int ti        = 0;

  while (t >= nt - ti)
  {
    t -= nt - ti;
    ++ti;
  }

  update_tile (a, off + ti * CH_NB, off + (ti + t) * CH_NB, Ls[0], Ls[1]);
}

// The factored diagonal blocks into S, and the lower triangle as the transpose
// of the factor (the backward sweep reads it row by row): one 64 x 64 tile per
// block, transposed through LDS.
__global__ void __launch_bounds__ (256)
k_potrf_finish (double *__restrict__ S, int np, const double *__restrict__ diagbuf)
{
  __shared__ double T[CH_NB][CH_NB + 1];
  const int nt  = (np + CH_NB - 1) / CH_NB;
  const int col = threadIdx.x & 63, w = threadIdx.x >> 6;
  int t = blockIdx.x, ti = 0;

  while (t >= nt - ti)
  {
    t -= nt - ti;
    ++ti;
  }

  const int r0 = ti * CH_NB, c0 = (ti + t) * CH_NB;

  if (t == 0)
  {
    const double *D = diagbuf + (size_t) ti * CH_NB * CH_NB;

    for (int r = w; r < CH_NB; r += 4)
      T[r][col] = (col >= r) ? D[r * CH_NB + col] : 0.0;
  }
  else
  {
    for (int r = w; r < CH_NB; r += 4)
      T[r][col] = (c0 + col < np) ? S[(size_t) (r0 + r) * np + c0 + col] : 0.0;
  }

  __syncthreads ();

  for (int r = w; r < CH_NB; r += 4)
  {
    if (t == 0)
    {
      if (r0 + r < np && r0 + col < np)
        S[(size_t) (r0 + r) * np + r0 + col] = (col >= r) ? T[r][col] : T[col][r];
    }
    else if (c0 + r < np)
    {
      S[(size_t) (c0 + r) * np + r0 + col] = T[col][r];
    }
  }
}

static void
potrf_step (double *S, int np, int kb, bool upd, int row_end, double *b, int *info, double *diagbuf, hipStream_t s)
{
  const int rest = np - kb - CH_NB;
  const int off  = kb + CH_NB;
  StepArgs a;

  a.S       = S;
  a.np      = np;
  a.kb      = kb;
  a.upd     = upd;
  a.info    = info;
  a.Ud      = diagbuf + (size_t) (kb / CH_NB) * CH_NB * CH_NB;
  a.b       = b;
  a.npb     = (rest > 0) ? (rest + CH_NB - 1) / CH_NB : 1;
  a.nrb     = (kb > 0 && rest > 0) ? (rest + 255) / 256 : 0;
  a.ntiles  = 0;

  if (upd && rest > 0 && row_end > off)
  {
    const int nt = (np - off + CH_NB - 1) / CH_NB;
    const int nr = (row_end - off + CH_NB - 1) / CH_NB;

    a.ntiles = nr * nt - nr * (nr - 1) / 2;
  }

  hipLaunchKernelGGL (k_potrf_step, dim3 (a.npb + a.nrb + (a.ntiles + 7) / 8 * 8), dim3 (256), 0, s, a);
}

// S = U^T U and y = U^{-T} b (in place).  While more than SP_MIN columns
// remain, four panels form a super-panel: each panel's update touches only
// the super-panel's own rows, and the rest of the trailing matrix gets one
// rank-256 update (a 4x shorter stream over it).  *info is the 1-based
// failing pivot, 0 on success; S and b are then not usable.
hipError_t
launch_potrf (double *S, int np, double *b, int *info, double *diagbuf, hipStream_t s)
{
  bool upd = false;

  for (int kb = 0; kb < np;)
  {
    if (!upd && np - kb > SP_MIN)
    {
      const int ke = kb + SP_NB;

      for (int kp = kb; kp < ke; kp += CH_NB)
        potrf_step (S, np, kp, kp > kb, ke, b, info, diagbuf, s);

      const hipError_t e = launch_trailing_update (S, np, SP_NB, ke, kb, s);

      if (e != hipSuccess)
        return e;

      kb = ke;
      continue;
    }

    potrf_step (S, np, kb, upd, np, b, info, diagbuf, s);
    upd = true;
    kb += CH_NB;
  }

  const int nt = (np + CH_NB - 1) / CH_NB;

  hipLaunchKernelGGL (k_potrf_finish, dim3 ((unsigned) ((size_t) nt * (nt + 1) / 2)), dim3 (256), 0, s, S, np,
                      diagbuf);

  return hipGetLastError ();
}

size_t
potrf_diag_doubles (int np)
{
  return (size_t) ((np + CH_NB - 1) / CH_NB) * CH_NB * CH_NB;
}

} // namespace nck

// Blocked Gauss-Jordan inverse without pivoting, bitwise equal to MATINV
// (PREP/template/GLOBAL/src/prep_GLOBAL.f90:516-568) for matrices too large
// for LDS (order n up to a few thousand), batched over `count` matrices.
//
// MATINV gives every element one fixed sequence of operations.  Forward
// step i (rows below i) and backward step i (rows above i) each replace
// element (r, j) by  B(r,j) - b(r) * B(i,j)  with the multiplier b(r) the
// value element (r, i) held just before the step (and element (r, i) itself
// first set to zero).  The pivot row i is final when the step reads it.  So
// the steps can be grouped in panels of KB consecutive pivots, provided each
// element still receives its updates one at a time in pivot order:
//
//   forward, panels up:
//     mb_panel_kernel   the panel's rows: the steps among them
//     mb_rows_kernel    every row below: the multipliers of the panel's KB
//                       steps from its panel columns, then the KB ordered
//                       updates of its columns
//   backward, panels up:
//     mb_rows_kernel    every row above, and the panel's own rows: row r of
//                       the panel takes its steps above r only, and the rows
//                       these read are the forward ones, so its rows do not
//                       wait for one another
//
// Rq holds the rows the steps read and Cq the panel's columns of the rows
// they change, both copied before a launch that overwrites them in place.
//
// A matrix is a chain of 3 n / KB launches, each bound by its latencies and
// dependent steps, not by the arithmetic, so work is repeated rather than
// handed over (every wavefront of the panel kernel eliminates the diagonal
// block for itself, every tile of the rows kernel forms its rows'
// multipliers), and the loops stay rolled: straight-line code of these steps
// (32 KB) was fetched more slowly than it ran.  Order 720 takes 1.0 ms a
// matrix, order 1440 2.7 (3.6 and 7.3 with five launches a panel).
//
// No operation is reassociated or fused (the file is built with
// -ffp-contract=off), so the result is bitwise MATINV's.
#include "sevp_dev.h"
#include "sevp_internal.h"

namespace sevp {

#define BM(i, j) B[(long)(i) + (long)(j) * n]  // 0-based, column-major

// Forward panel [p0, p0 + kb).  Workgroups [0, ncol): the panel's steps on 64
// columns, with the diagonal block eliminated in every workgroup.
//   * Wavefronts 0-3 hold the diagonal block (thread (r, g): row r, columns
//     g, g + 8, ...).  Step i: row i is scaled by its reciprocal pivot, the
//     rows after it take  B(r,c) <- (c == i ? 0 : B(r,c)) - m B(i,c), m =
//     B(r,i); the next step's row and column go to LDS, one barrier a step.
//   * Wavefront 4 holds the columns, one a lane, its rows in registers (read
//     and written through LDS, so that the column-major matrix moves in runs).
//     It is one step behind: the multipliers of step i (column i of the
//     block) are requested while step i - 1 is made.  After a step the rows
//     move up one place, so the loop stays rolled.
// A step is its chain: LDS reads, the division, the update, the barrier.  One
// wavefront doing both parts, with the multipliers as scalar operands, took
// 15 us for the 32 steps; this takes 9.5.
// Rows past kb are those of a unit matrix: they change nothing and are not
// stored.  Every workgroup reads the diagonal block, so the first one leaves
// its result in Cq's rows of the panel (column c at Cq[c n + p0 ..]) and the
// rows kernel puts it in place.  The other workgroups copy the panel's
// columns of the rows below to Cq[k n + r].
constexpr int MP_THREADS = 320;

// Steps i0 .. i0 + 7 of wavefront 4, whose live rows are y[0 .. NR - 1].
// m: the multipliers of step i (row i + 1 + r at m[r]), d its pivot.
template <int NR>
__device__ __forceinline__ void panel_cols(double (&y)[MB_KB], double (&m)[MB_KB], double &d, int i0,
                                           const double (*col)[2 * MB_KB], double *xs) {
#pragma unroll 1
  for (int i4 = i0; i4 < i0 + 8; i4 += 4) {
    unroll<0, 4>([&](auto U) {
      constexpr int u = decltype(U)::value;
      __syncthreads();  // column i + 1 is in LDS
      double mn[NR];
      const double *cn = col[(u + 1) & 3] + i4 + u + 1;
      const double dn = cn[0];
#pragma unroll
      for (int r = 0; r + 1 < NR; ++r) mn[r] = cn[r + 1];
      const double f = y[0] * (1.0 / d);
      xs[i4 + u] = f;
#pragma unroll
      for (int r = 0; r + 1 < NR; ++r) y[r] = y[r + 1] - m[r] * f;
#pragma unroll
      for (int r = 0; r + 1 < NR; ++r) m[r] = mn[r];
      d = dn;
    });
  }
}

__global__ __launch_bounds__(MP_THREADS) void mb_panel_kernel(double *mats, long ms, int n, int p0,
                                                              int kb, int ncol, double *rqs,
                                                              double *cqs, long qs, int *zp) {
  __shared__ double Xs[64][MB_KB + 1];
  __shared__ double rowb[4][MB_KB];      // row i of the block before step i, at i % 4
  __shared__ double colb[4][2 * MB_KB];  // column i; past row 31: never used
  double *B = mats + (long)blockIdx.y * ms;
  double *Rq = rqs + (long)blockIdx.y * qs;
  double *Cq = cqs + (long)blockIdx.y * qs;
  const int t = threadIdx.x, b = blockIdx.x;
  if (b >= ncol) {
    for (int idx = t; idx < 64 * kb; idx += MP_THREADS) {
      const int r = p0 + kb + 64 * (b - ncol) + (idx & 63), k = idx >> 6;
      if (r < n) Cq[(long)k * n + r] = BM(r, p0 + k);
    }
    return;
  }
  if (t < 4 * MB_KB) colb[t / MB_KB][MB_KB + t % MB_KB] = 0.0;
  if (t < 256) {
    const int r = t >> 3, g = t & 7;
    double a[4];  // a[s]: column g + 8 ((s + i / 8) % 4), so that step i's column is in a[0]
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = g + 8 * s;
      const double v = BM(p0 + min(r, kb - 1), p0 + min(c, kb - 1));
      a[s] = (r < kb && c < kb) ? v : (r == c ? 1.0 : 0.0);
    }
    int off[4] = {g, g + 8, g + 16, g + 24};
    int zeros = 0;
    if (r == 0)
#pragma unroll
      for (int s = 0; s < 4; ++s) rowb[0][off[s]] = a[s];
    if (g == 0) colb[0][r] = a[0];
    __syncthreads();
#pragma unroll 1
    for (int i8 = 0; i8 < MB_KB; i8 += 8) {
      unroll<0, 8>([&](auto U) {
        constexpr int u = decltype(U)::value;
        const int i = i8 + u;
        const double d = rowb[u & 3][i], m = colb[u & 3][r];
        double e[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) e[s] = rowb[u & 3][off[s]];
        __builtin_amdgcn_sched_barrier(0);  // every read before the division waits
        const double piv = 1.0 / d;
        const bool mine = g == u, below = r > i, own = r == i;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          double es = e[s], as = a[s];
          if (s == 0) {
            es = mine ? 1.0 : es;
            as = mine ? 0.0 : as;
          }
          es = es * piv;
          const double v = as - m * es;
          a[s] = below ? v : (own ? es : a[s]);
        }
        zeros += (d == 0.0 && i < kb);
        if (u == 7) {  // the next step's column moves to a[0]
          const double w = a[0];
          const int o = off[0];
          a[0] = a[1]; a[1] = a[2]; a[2] = a[3]; a[3] = w;
          off[0] = off[1]; off[1] = off[2]; off[2] = off[3]; off[3] = o;
        }
        if (r == i + 1)
#pragma unroll
          for (int s = 0; s < 4; ++s) rowb[(u + 1) & 3][off[s]] = a[s];
        if (g == ((u + 1) & 7)) colb[(u + 1) & 3][r] = a[0];
        __syncthreads();
      });
    }
    if (b == 0 && r < kb)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int c = g + 8 * s;
        if (c < kb) {
          Rq[(long)r * n + p0 + c] = a[s];
          Cq[(long)c * n + p0 + r] = a[s];
        }
      }
    if (b == 0 && t == 0 && zeros && zp) atomicAdd(zp, zeros);
    return;
  }
  const int lane = t & 63, c = lane & 31, h = lane >> 5;
  {
    double v[MB_KB];
    const int k = min(c, kb - 1);
#pragma unroll
    for (int q = 0; q < MB_KB; ++q) v[q] = BM(p0 + k, min(64 * b + 2 * q + h, n - 1));
#pragma unroll
    for (int q = 0; q < MB_KB; ++q) Xs[2 * q + h][c] = c < kb ? v[q] : 0.0;
  }
  wave_lds_sync();
  double y[MB_KB], m[MB_KB], d;
#pragma unroll
  for (int k = 0; k < MB_KB; ++k) y[k] = Xs[lane][k];
  __syncthreads();  // column 0 is in LDS
  d = colb[0][0];
#pragma unroll
  for (int r = 0; r + 1 < MB_KB; ++r) m[r] = colb[0][r + 1];
  panel_cols<32>(y, m, d, 0, colb, Xs[lane]);
  panel_cols<24>(y, m, d, 8, colb, Xs[lane]);
  panel_cols<16>(y, m, d, 16, colb, Xs[lane]);
  panel_cols<8>(y, m, d, 24, colb, Xs[lane]);
  wave_lds_sync();
#pragma unroll
  for (int q = 0; q < MB_KB; ++q) {
    const int cc = 64 * b + 2 * q + h;
    if (c < kb && cc < n && (cc < p0 || cc >= p0 + kb)) BM(p0 + c, cc) = Xs[2 * q + h][c];
  }
  const int j = 64 * b + lane;
  if (j < n && (j < p0 || j >= p0 + kb))
    for (int k = 0; k < kb; ++k) Rq[(long)k * n + j] = Xs[lane][k];
}

// The panel's steps on the rows [r_lo, r_hi), in tiles of 64 by 16 CT
// columns.  Four lanes a row form its multipliers (lane q holds its panel
// columns q, q + 4, ...: step k's is column k's value then, handed to the row
// by a quad broadcast; a column that has given its multiplier is moved out),
// then every thread makes the ordered updates of its 4 CT elements.  A column
// j of the panel starts from zero at step j, and, backward, row r of the panel
// from its element at step r + 1.
// Forward, one more row of workgroups puts the diagonal block in place.
// Backward, it copies the next panel's rows to Rq's other half, and the tiles
// leave the next panel's columns in Cq's other half (next: offset of the
// other halves, 0 for the last panel).
constexpr int MT_R = 64;
template <int CT, bool BACK>
__global__ __launch_bounds__(256) void mb_rows_kernel(double *mats, long ms, int n, int p0, int kb,
                                                      int r_lo, int r_hi, double *rqs, double *cqs,
                                                      long qs, long next) {
  constexpr int TC = 16 * CT;
  __shared__ double D[MB_KB + 1][2 * MB_KB + 1];  // past column kb and row 31: never used
  __shared__ double Ms[MT_R][MB_KB + 1];
  __shared__ double Rs[MB_KB][TC + 1];
  double *B = mats + (long)blockIdx.z * ms;
  double *Rq = rqs + (long)blockIdx.z * qs;
  double *Cq = cqs + (long)blockIdx.z * qs;
  const int t = threadIdx.x;
  const int p1 = p0 + kb;
  if (blockIdx.y == gridDim.y - 1) {
    if (!BACK) {
      if (blockIdx.x == 0)
        for (int idx = t; idx < kb * kb; idx += 256) {
          const int r = idx % kb, c = idx / kb;
          BM(p0 + r, p0 + c) = Cq[(long)c * n + p0 + r];
        }
    } else if (next) {
      const int kn = min(MB_KB, n - p1);
      for (long idx = blockIdx.x * 256 + t; idx < (long)kn * n; idx += 256 * gridDim.x) {
        const int k = (int)(idx % kn), j = (int)(idx / kn);
        Rq[next + (long)k * n + j] = BM(p1 + k, j);
      }
    }
    return;
  }
  const int r0 = r_lo + blockIdx.x * MT_R, c0 = blockIdx.y * TC;
  const int row = t >> 2, q = t & 3;
  const int rr = min(r0 + row, r_hi - 1);
  const bool own = BACK && rr >= p0;  // a row of the panel
  double cur[MB_KB / 4];
#pragma unroll
  for (int s = 0; s < MB_KB / 4; ++s) {
    const int k = min(4 * s + q, kb - 1);
    cur[s] = own ? Rq[(long)(rr - p0) * n + p0 + k] : Cq[(long)k * n + rr];
  }
  const int tr = t % 16, tc = t / 16;  // rows tr + 16 i, columns CT tc + jj
  double acc[4][CT];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int jj = 0; jj < CT; ++jj)
      acc[i][jj] = BM(min(r0 + tr + 16 * i, r_hi - 1), min(c0 + CT * tc + jj, n - 1));
  for (int idx = t; idx < MB_KB * 2 * MB_KB; idx += 256) {
    const int k = idx / (2 * MB_KB), j = idx % (2 * MB_KB);
    D[k][j] = j < kb ? Rq[(long)min(k, kb - 1) * n + p0 + j] : 0.0;
  }
  for (int idx = t; idx < MB_KB * TC; idx += 256) {
    const int k = idx / TC, cc = idx % TC;
    Rs[k][cc] = Rq[(long)min(k, kb - 1) * n + min(c0 + cc, n - 1)];
  }
  __syncthreads();
  const int first = own ? rr - p0 + 1 : 0;  // this row's first step
  {
    // each step's row of D is requested a step ahead
    const double *dp = &D[0][q];
    double dv[MB_KB / 4];
#pragma unroll
    for (int s = 0; s < MB_KB / 4; ++s) dv[s] = dp[4 * s];
#pragma unroll 1
    for (int k4 = 0; k4 < kb; k4 += 4) {
      unroll<0, 4>([&](auto KI) {
        constexpr int ki = decltype(KI)::value;
        const int k = k4 + ki;  // past kb: steps that no one uses
        dp += 2 * MB_KB + 1 + (ki == 3 ? 4 : 0);
        double dn[MB_KB / 4];
#pragma unroll
        for (int s = 0; s < MB_KB / 4; ++s) dn[s] = dp[4 * s];
        const double bk = quad_bcast<ki>(cur[0]);
        if (q == ki) Ms[row][k] = bk;
#pragma unroll
        for (int s = 0; s < MB_KB / 4; ++s) {
          const double v = cur[s] - bk * dv[s];
          cur[s] = (BACK && k < first) ? cur[s] : v;
          dv[s] = dn[s];
        }
      });
#pragma unroll
      for (int s = 0; s + 1 < MB_KB / 4; ++s) cur[s] = cur[s + 1];
    }
  }
  __syncthreads();
  const bool crosses = (c0 < p1 && c0 + TC > p0) || (BACK && r0 + MT_R > p0);
  if (!crosses) {
#pragma unroll 4
    for (int k = 0; k < kb; ++k) {
      double mv[4], rv[CT];
#pragma unroll
      for (int i = 0; i < 4; ++i) mv[i] = Ms[tr + 16 * i][k];
#pragma unroll
      for (int jj = 0; jj < CT; ++jj) rv[jj] = Rs[k][CT * tc + jj];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jj = 0; jj < CT; ++jj) acc[i][jj] = acc[i][jj] - mv[i] * rv[jj];
    }
  } else {
    int from[4][CT];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jj = 0; jj < CT; ++jj) {
        const int r = r0 + tr + 16 * i, c = c0 + CT * tc + jj;
        const int f = (BACK && r >= p0) ? r - p0 + 1 : 0;
        const bool in = c >= p0 + f && c < p1;  // its own step is one of the row's
        from[i][jj] = in ? c - p0 : f;
        acc[i][jj] = in ? 0.0 : acc[i][jj];
      }
#pragma unroll 4
    for (int k = 0; k < kb; ++k) {
      double mv[4], rv[CT];
#pragma unroll
      for (int i = 0; i < 4; ++i) mv[i] = Ms[tr + 16 * i][k];
#pragma unroll
      for (int jj = 0; jj < CT; ++jj) rv[jj] = Rs[k][CT * tc + jj];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jj = 0; jj < CT; ++jj) {
          const double v = acc[i][jj] - mv[i] * rv[jj];
          acc[i][jj] = k >= from[i][jj] ? v : acc[i][jj];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int jj = 0; jj < CT; ++jj) {
      const int r = r0 + tr + 16 * i, c = c0 + CT * tc + jj;
      if (r < r_hi && c < n) {
        BM(r, c) = acc[i][jj];
        if (BACK && next && c >= p1 && c < p1 + MB_KB) Cq[next + (long)(c - p1) * n + r] = acc[i][jj];
      }
    }
}

// Rq(k, j) = B(k, j), k < kb: the first panel's rows for the backward steps.
__global__ void mb_copy_rows_kernel(const double *mats, long ms, int n, int kb, double *rqs, long qs) {
  const double *B = mats + (long)blockIdx.y * ms;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < (long)kb * n) rqs[(long)blockIdx.y * qs + (t % kb) * n + t / kb] = BM((int)(t % kb), (int)(t / kb));
}
#undef BM

hipError_t launch_matinv_blocked(double *mats, long ms, int n, int count, int *zp,
                                 double *scratch, hipStream_t st) {
  const long half = (long)MB_KB * n, qs = 4 * half;
  double *rq = scratch, *cq = scratch + 2 * half;
  const int ncol = (n + 63) / 64;
  // 64-column tiles repeat the multipliers less often, 32-column ones fill
  // the GPU: the wider where there are enough of them
  auto rows = [&](bool back, int p0, int kb, int r_lo, int r_hi, int cur, long next) {
    const int tiles = (r_hi - r_lo + MT_R - 1) / MT_R;
    const bool wide = (long)tiles * ((n + 63) / 64) * count >= 256;
    const int tcol = wide ? 64 : 32;
    const dim3 grid(tiles > 0 ? tiles : 1, (r_hi > r_lo ? (n + tcol - 1) / tcol : 0) + 1, count);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, mats, ms, n, p0, kb, r_lo, r_hi,
                         rq + cur * half, cq + cur * half, qs, next);
    };
    if (back) wide ? go(mb_rows_kernel<4, true>) : go(mb_rows_kernel<2, true>);
    else wide ? go(mb_rows_kernel<4, false>) : go(mb_rows_kernel<2, false>);
  };
  for (int p0 = 0; p0 < n; p0 += MB_KB) {
    const int p1 = min(n, p0 + MB_KB), kb = p1 - p0;
    hipLaunchKernelGGL(mb_panel_kernel, dim3(ncol + (n - p1 + 63) / 64, count), dim3(MP_THREADS), 0, st, mats,
                       ms, n, p0, kb, ncol, rq, cq, qs, zp);
    rows(false, p0, kb, p1, n, 0, 0);
  }
  {
    const int kb = min(n, MB_KB);
    hipLaunchKernelGGL(mb_copy_rows_kernel, dim3((unsigned)(((long)kb * n + 255) / 256), count),
                       dim3(256), 0, st, mats, ms, n, kb, rq, qs);
  }
  for (int q0 = 0, cur = 0; q0 < n; q0 += MB_KB, cur ^= 1) {
    const int q1 = min(n, q0 + MB_KB);
    rows(true, q0, q1 - q0, 0, q1, cur, q1 < n ? (cur ? -half : half) : 0);
  }
  return hipGetLastError();
}

}  // namespace sevp

// Full-width SEVP building blocks (REP1, REP, PRE1, PRE and the strip PRE),
// batched over independent right-hand sides / unit vectors.
//
// March kernels use trapezoid tiles: a wavefront marches 64*K consecutive
// columns (K per lane, east/west neighbours through DPP wave shifts), and
// after s rows only the columns at least s away from the tile edge are still
// exact, so each tile carries `halo` extra columns on each side and writes
// only its central `tile_out` columns.  Recomputing the halo columns repeats
// exactly the same operations on exactly the same operands, so the written
// values are bitwise those of a march over the whole width.  Periodic
// problems index columns modulo the width; this reproduces the reference's
// halo copies X(1)=X(I0-1), X(I0)=X(2), which only ever duplicate interior
// values, and a final pass (halo_fix_kernel) leaves the halo columns as the
// reference leaves them.
//
// The correction products keep every output one sequential sum over k from
// zero with separately rounded multiply and add: the reference's
// DUM2(N)=DUM2(N)+DUM1(M)*RINV(M,N) loop order.
//
// MATINV is the reference's Gauss-Jordan without pivoting
// (PREP/template/GLOBAL/src/prep_GLOBAL.f90:516-568) with the matrix held in
// LDS when it fits (larger orders use the blocked form in sevp_matinv.hip);
// each element receives the same sequence of operations as in the reference,
// only the independent element updates of one step run in parallel.
#include <hip/hip_ext.h>

#include "sevp_dev.h"
#include "sevp_internal.h"
#include "sevp_march.h"
#include "sevp_tiles.h"

namespace sevp {

template <int K, int MODE>
__global__ __launch_bounds__(64) void march_kernel(MarchArgs p) {
  march_body<K, MODE>(p, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, threadIdx.x);
}

// Choose lanes-per-column K and the tile size for a march of `steps` rows.
static void march_shape(int w, int steps, int &K, int &tile, int &halo, int &ntiles) {
  halo = steps + 1;
  int best = -1;
  long bestcost = 0;
  for (int k : {1, 2, 4}) {
    const int t = 64 * k - 2 * halo;
    if (t <= 0) continue;
    const long n = (w + t - 1) / t;
    const long cost = n * k;
    if (best < 0 || cost < bestcost) {
      best = k;
      bestcost = cost;
      tile = t;
      ntiles = (int)n;
    }
  }
  K = best;
}

template <int MODE>
static hipError_t launch_march_mode(const MarchArgs &a0, int nbatch, int nstrips, hipStream_t st) {
  MarchArgs a = a0;
  int K, tile, halo, ntiles;
  march_shape(a.w, a.jf - a.js + 1, K, tile, halo, ntiles);
  if (K < 0) return hipErrorInvalidValue;
  a.tile_out = tile;
  a.halo = halo;
  dim3 grid(ntiles, nbatch, nstrips);
  if (K == 1) hipLaunchKernelGGL((march_kernel<1, MODE>), grid, dim3(64), 0, st, a);
  else if (K == 2) hipLaunchKernelGGL((march_kernel<2, MODE>), grid, dim3(64), 0, st, a);
  else hipLaunchKernelGGL((march_kernel<4, MODE>), grid, dim3(64), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_march(int mode, const MarchArgs &a, int nbatch, hipStream_t st) {
  const int nstrips = (mode == MODE_PRE) ? a.nrhs : 1;  // PRE: nrhs carries the strip count
  if (mode == MODE_PART) return launch_march_mode<MODE_PART>(a, nbatch, 1, st);
  if (mode == MODE_HOM) return launch_march_mode<MODE_HOM>(a, nbatch, 1, st);
  return launch_march_mode<MODE_PRE>(a, nbatch, nstrips, st);
}

// Closure residual of equation row ieb-1 at column c (1-based) for RHS r,
// given row ieb's west/centre/east values and row ieb+1's value at c.
__device__ __forceinline__ double closure_resid(const ResidArgs &p, int r, int c, const double *x,
                                                double west, double center, double east,
                                                double north) {
  const int i0 = p.i2 + 2, jr = p.ieb - 1;
  const long co = (long)(c - 1) + (long)(jr - 1) * p.i2;
  const double fv = p.f64 ? p.f64[(long)r * p.f_stride + co] : (double)p.f[(long)r * p.f_stride + co];
  return fv - (double)p.ax[co] * west - (double)p.ay[co] * x[f2(i0, c + 1, jr)] -
         (double)p.bb[co] * center - (double)p.cx[co] * east - (double)p.cy[co] * north;
}

// West and east neighbours in row ieb of column c, reading row values
// through rowv (which applies the DUM0 restore where there is one).
template <class RowV>
__device__ __forceinline__ void row_nbrs(const ResidArgs &p, const double *x, int c, RowV rowv,
                                         double &west, double &east) {
  const int i2 = p.i2, i0 = i2 + 2, ieb = p.ieb;
  if (p.periodic) {
    west = rowv(c == 1 ? i2 : c - 1);
    east = rowv(c == i2 ? 1 : c + 1);
  } else {
    west = (c == 1) ? x[f2(i0, 1, ieb)] : rowv(c - 1);
    east = (c == i2) ? x[f2(i0, i0, ieb)] : rowv(c + 1);
  }
}

// Backward restore of X(:, ieb) from DUM0 and closure residual at row ieb-1.
__device__ void resid_body(const ResidArgs &p, long t) {
  if (t >= (long)p.nrhs * p.i2) return;
  const int r = (int)(t / p.i2);
  const int c = (int)(t % p.i2) + 1;
  const int i2 = p.i2, i0 = i2 + 2, ieb = p.ieb;
  double *x = p.x + (long)r * p.x_stride;
  const double *d0 = p.dum0 ? p.dum0 + (long)r * p.dum0_stride + (long)(p.nb - 1) * i2 : nullptr;
  auto rowv = [&](int cc) -> double {  // value of row ieb at column cc (1..i2) after the restore
    return d0 ? d0[cc - 1] : x[f2(i0, cc + 1, ieb)];
  };
  const double center = rowv(c);
  double west, east;
  row_nbrs(p, x, c, rowv, west, east);
  const double e = closure_resid(p, r, c, x, west, center, east, x[f2(i0, c + 1, ieb + 1)]);
  if (p.e) p.e[(long)r * i2 + c - 1] = e;
  if (p.e32) p.e32[(long)r * i2 + c - 1] = (float)e;
  if (d0) x[f2(i0, c + 1, ieb)] = center;
}

// Mixed-precision backward, per (rhs, column): X(apply_row) += the free-row
// correction of the block above (summed from its partial products), then,
// when do_resid, the closure residual of the block below (row ieb-1 =
// apply_row-2), whose only read of apply_row is this column's.  X(ieb) was
// never overwritten by the forward pass here, so no restore is needed.
__device__ void apply_resid_body(const ResidArgs &p, long t) {
  if (t >= (long)p.nrhs * p.i2) return;
  const int r = (int)(t / p.i2);
  const int c = (int)(t % p.i2) + 1;
  const int i2 = p.i2, i0 = i2 + 2, ieb = p.ieb;
  double *x = p.x + (long)r * p.x_stride;
  const long xa = f2(i0, c + 1, p.apply_row);
  const double north = x[xa] + p.corr.sum(r, c - 1);
  x[xa] = north;
  if (!p.do_resid) return;
  auto rowv = [&](int cc) -> double { return x[f2(i0, cc + 1, ieb)]; };
  double west, east;
  row_nbrs(p, x, c, rowv, west, east);
  const double e = closure_resid(p, r, c, x, west, rowv(c), east, north);
  if (p.e) p.e[(long)r * i2 + c - 1] = e;
  if (p.e32) p.e32[(long)r * i2 + c - 1] = (float)e;
}

__global__ void resid_kernel(ResidArgs p) {
  resid_body(p, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// The backward H march of block b and the restore + closure residual of
// block b-1 touch disjoint rows and read nothing the other writes: one
// launch runs both (march tiles first, then 64-column residual groups).
template <int K>
__device__ __forceinline__ void hom_resid_body(const MarchArgs &m, const ResidArgs &r, int ntiles,
                                               int has_resid, long b) {
  const long nm = (long)ntiles * m.nrhs;
  if (b < nm) {
    march_body<K, MODE_HOM>(m, (int)(b % ntiles), (int)(b / ntiles), 0, 1, threadIdx.x);
    return;
  }
  if (!has_resid) return;
  if (r.corr.on()) apply_resid_body(r, (b - nm) * 64 + threadIdx.x);
  else resid_body(r, (b - nm) * 64 + threadIdx.x);
}

template <int K>
__global__ __launch_bounds__(64) void hom_resid_kernel(MarchArgs m, ResidArgs r, int ntiles,
                                                       int has_resid) {
  hom_resid_body<K>(m, r, ntiles, has_resid, blockIdx.x);
}

int march_tiles(MarchArgs &a, int K) {
  const int steps = a.jf - a.js + 1;
  int k, tile, halo, ntiles;
  march_shape(a.w, steps, k, tile, halo, ntiles);
  if (k < 0) return 0;
  if (K > 0) {  // a given lane width (any width whose tile is positive gives the same values)
    tile = 64 * K - 2 * halo;
    if (tile <= 0) return 0;
    ntiles = (a.w + tile - 1) / tile;
  }
  a.tile_out = tile;
  a.halo = halo;
  return ntiles;
}

int march_lanes(int w, int steps) {
  int k, tile, halo, ntiles;
  march_shape(w, steps, k, tile, halo, ntiles);
  return k;
}

long hom_resid_prepare(const MarchArgs &a0, const ResidArgs *r, int K, HomResidEnt &ent) {
  ent.m = a0;
  const int ntiles = march_tiles(ent.m, K);
  if (ntiles <= 0) return -1;
  ent.ntiles = ntiles;
  const long nm = (long)ntiles * a0.nrhs;
  const long nr = r ? ((long)r->nrhs * r->i2 + 63) / 64 : 0;
  const bool march = a0.jf >= a0.js;
  ent.r = r ? *r : ResidArgs{};
  ent.has_resid = r != nullptr;
  if (!march) ent.m.nrhs = 0;  // no march blocks: every block is a residual group
  return (march ? nm : 0) + nr;
}

hipError_t launch_hom_resid(const MarchArgs &a0, const ResidArgs *r, hipStream_t st) {
  const int K = march_lanes(a0.w, a0.jf - a0.js + 1);
  if (K < 0) return hipErrorInvalidValue;
  HomResidEnt e;
  const long nwg = hom_resid_prepare(a0, r, K, e);
  if (nwg < 0) return hipErrorInvalidValue;
  if (nwg == 0) return hipSuccess;
  const dim3 grid((unsigned)nwg);
  if (K == 1) hipLaunchKernelGGL((hom_resid_kernel<1>), grid, dim3(64), 0, st, e.m, e.r, e.ntiles, e.has_resid);
  else if (K == 2) hipLaunchKernelGGL((hom_resid_kernel<2>), grid, dim3(64), 0, st, e.m, e.r, e.ntiles, e.has_resid);
  else hipLaunchKernelGGL((hom_resid_kernel<4>), grid, dim3(64), 0, st, e.m, e.r, e.ntiles, e.has_resid);
  return hipGetLastError();
}

hipError_t launch_resid(const ResidArgs &a, hipStream_t st) {
  const long n = (long)a.nrhs * a.i2;
  hipLaunchKernelGGL(resid_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Sequential-order FP64 products: every output is one thread's sum over k
// from zero, in order, with separately rounded multiply and add.

// The correction products of a solve, D(m, n) = sum_k A(m, k) B(k, n), both
// operands with consecutive k adjacent (the error rows and a column-major
// influence matrix), with fused epilogues.
//
// A computing wavefront holds 16 right-hand sides (the lanes of a row) by 4
// columns (its four 16-lane rows), one sum a lane.  A lane's B values are its
// column's, so a row of lanes holds 32 consecutive k of the column, two a
// lane, and each k reaches the row by a DPP broadcast; only A is read from
// LDS per term (16 bytes for two k).  An output and k cost 8 bytes of LDS
// reads, half of what a tile that reads both operands from LDS costs, which
// bounded such a kernel.  The multiply of a term does not depend on the sum:
// the terms of the next 8 k are formed between the additions of these.  What
// bounds it now is LDS all the same (97 to 109 bytes a clock and CU at 64
// right-hand sides): 21 clocks a term; 64 right-hand sides at 960 columns
// take 13.3 us (22.5 before), 32 at 1440 columns 17.7 us (32 before).
//
// A matrix comes from HBM once a solve, so a launch is that latency and its
// sums.  NL loading wavefronts stream both operands into LDS with DMAs
// (global_load_lds: no registers and no waits while they fly), R chunks of
// 64 k ahead; a register ring of half that depth waited for HBM.  NW
// computing wavefronts side by side share A's chunks.  One barrier a chunk,
// in the middle of its sum, tells that the next chunk has landed and that the
// one before is no longer read, so neither side waits at a chunk's start.
// Past K both operands are zero in LDS: a sum that started from +0 keeps its
// bits when +0 is added.
constexpr int GS_K = 64;

// 16 or 4 bytes a lane of a 64-lane run at dst (wave-uniform) come from src.
__device__ __forceinline__ void load_lds16(const void *src, void *dst) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void *)(src),
                                   (__attribute__((address_space(3))) void *)(dst), 16, 0, 0);
}
__device__ __forceinline__ void load_lds4(const void *src, void *dst) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void *)(src),
                                   (__attribute__((address_space(3))) void *)(dst), 4, 0, 0);
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The chunk barrier: the side that writes LDS waits for its writes; the side
// that reads it has used what it read from the buffer that is written next,
// and its reads in flight are of another.
__device__ __forceinline__ void bar_written() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ void bar_reader() { asm volatile("s_barrier" ::: "memory"); }

// One workgroup's operand ring.  B: a computing wavefront's chunk is two
// runs of 64 pairs in the order its lanes use them.  A: the rows of a pair
// adjacent, so that the 16 rows' reads of one pair are one run.
template <int NW, int R>
struct SeqRing {
  double2 b[R][NW][2][64];
  double2 a[R][32][16];
};

// Loading wavefront `l` of NL: every NL-th of a chunk's DMAs.  W = 16: runs
// of pairs at 16-byte boundaries (an even K; the clamped pairs past K are
// whole pairs of the run).  W = 4: any boundary, each k clamped by itself.
template <int NW, int NL, int R, int W>
__device__ __forceinline__ void seq_load(const GemmArgs &p, SeqRing<NW, R> &S, int n0, int m0,
                                         int rows, int nlast, int l, int lane) {
  constexpr int PP = 16 / W;                             // DMAs of a run of 64 pairs
  constexpr int I = (2 * NW + 8) * PP, PER = I / NL;  // DMAs of a chunk; of this wavefront
  static_assert(I % NL == 0 && (R - 3) * PER <= 63, "the waits count this wavefront's DMAs");
  const double *run[PER];
  int off[PER];  // k of this lane's element in a chunk
  char *dst[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int id = l + NL * i, blk = id / PP, e = (id % PP) * 64 + lane;  // element of the run
    const int s = e / PP;                                                 // its pair's place
    if (blk < 2 * NW) {
      const int w = blk >> 1, q = blk & 1;
      run[i] = p.b + (long)min(n0 + 4 * w + (s >> 4), p.N - 1) * p.b_sn;
      off[i] = 32 * q + 2 * (s & 15);
      dst[i] = reinterpret_cast<char *>(&S.b[0][w][q][0]) + (id % PP) * 64 * W;
    } else {
      const int ps = (blk - 2 * NW) * 64 + s;
      run[i] = p.a + (long)(m0 + min(ps & 15, rows - 1)) * p.a_sm;
      off[i] = 2 * (ps >> 4);
      dst[i] = reinterpret_cast<char *>(&S.a[0][0][0]) + ((blk - 2 * NW) * 64 * PP + (id % PP) * 64) * W;
    }
  }
  auto issue = [&](int c, int slot) {
    const int k0 = c * GS_K;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int id = l + NL * i;
      char *d = dst[i] + (long)slot * (id / PP < 2 * NW ? sizeof(S.b[0]) : sizeof(S.a[0]));
      if constexpr (W == 16) {
        load_lds16(run[i] + min(k0 + off[i], p.K - 2), d);
      } else {
        const int comp = lane & 3;
        load_lds4(reinterpret_cast<const uint32_t *>(run[i] + min(k0 + off[i] + (comp >> 1), p.K - 1)) +
                      (comp & 1), d);
      }
    }
  };
  // the chunks issued after the one waited for (at most R - 3) may still fly
  auto landed = [&](int newer) {
    unroll<0, R - 2>([&](auto N) {
      constexpr int n = decltype(N)::value;
      if (newer == n) wait_loads<n * PER>();
    });
  };
  // zeros over what the last chunk's clamped addresses brought, past K
  auto zero_past = [&](int c, int slot) {
    if (c != nlast) return;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int id = l + NL * i;
      char *d = dst[i] + (long)slot * (id / PP < 2 * NW ? sizeof(S.b[0]) : sizeof(S.a[0])) + lane * W;
      const int k = c * GS_K + off[i];
      if constexpr (W == 16) {
        if (k >= p.K) *reinterpret_cast<double2 *>(d) = make_double2(0.0, 0.0);
      } else {
        if (k + ((lane & 3) >> 1) >= p.K) *reinterpret_cast<uint32_t *>(d) = 0u;
      }
    }
  };
  for (int c = 0; c < R && c <= nlast; ++c) issue(c, c);
  landed(min(nlast, R - 3));
  zero_past(0, 0);
  bar_written();
  int sn = 1;        // slot of chunk c + 1
  int slot = R - 1;  // of chunk c - 1 + R
  for (int c = 0; c < nlast; ++c) {
    landed(min(nlast - c - 1, R - 3));
    zero_past(c + 1, sn);
    bar_written();
    if (c >= 1 && c - 1 + R <= nlast) issue(c - 1 + R, slot);
    slot = slot + 1 == R ? 0 : slot + 1;
    sn = sn + 1 == R ? 0 : sn + 1;
  }
}

template <int NW, int NL, int R, int W>
__global__ __launch_bounds__(64 * (NW + NL)) void gemm_seq_kernel(GemmArgs p) {
  constexpr int NT = 4 * NW;  // columns of the tile
  __shared__ __align__(16) SeqRing<NW, R> S;
  __shared__ double Ts[16][NT + 1];
  span_begin(p.tspan);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // XCD-aware placement: the dispatcher deals workgroups to the 8 XCDs in
  // turn, so the row tiles of one column tile get ids on the same XCD, one
  // after another, and read that tile of B from HBM once (the others from
  // the XCD's L2); ids past the last column tile have no tile
  const int ntn = (p.N + NT - 1) / NT, nmb = (p.M + 15) / 16;
  const int slot = blockIdx.x >> 3, tcol = (slot / nmb) * 8 + (blockIdx.x & 7);
  if (tcol >= ntn) {
    span_end(p.tspan);
    return;
  }
  const int n0 = tcol * NT, m0 = (slot % nmb) * 16;
  const int K = p.K, rows = min(16, p.M - m0);
  const int nlast = (K + GS_K - 1) / GS_K - 1;  // the chunks before it are whole
  if (wave >= NW) {
    seq_load<NW, NL, R, W>(p, S, n0, m0, rows, nlast, wave - NW, lane);
    __syncthreads();  // the computing wavefronts' sums are in Ts
    span_end(p.tspan);
    return;
  }
  // the epilogue's element (em, en) of this thread and its operands, which
  // do not depend on the product (threads without one load the tile's first)
  const bool eok = m0 + t / NT < p.M && n0 + t % NT < p.N;
  const int em = eok ? m0 + t / NT : m0, en = eok ? n0 + t % NT : n0;
  double xv = 0.0;
  float cyv = 0.f;
  double *ex = nullptr;
  if (p.ep != EP_CPL) {
    ex = p.x + (long)em * p.x_stride + f2(p.i2 + 2, en + 2, p.xrow);
    xv = *ex;
    if (p.g) cyv = p.cy[(long)en + (long)(p.cyrow - 1) * p.i2];
  }
  // A chunk's sum runs in eight groups of 8 k.  Before group g is added, A's
  // values of group g + 2 are requested, and the products of group g + 1 are
  // formed between its additions; the last two groups do so for the next
  // chunk (slot sn).
  const double2 *ab = &S.a[0][0][lane & 15];
  const double2 *bb = &S.b[0][wave][0][lane];
  double acc = 0.0, pr[2][8];
  double2 av[2][4], bv[2], bn[2];
  auto read_a = [&](int sl, auto G) {
    constexpr int g = decltype(G)::value;
#pragma unroll
    for (int j = 0; j < 4; ++j) av[g & 1][j] = ab[sl * (32 * 16) + (4 * g + j) * 16];
  };
  auto read_b = [&](int sl, double2 (&b_)[2]) {
    const double2 *q = bb + sl * (sizeof(S.b[0]) / 16);
    b_[0] = q[0];
    b_[1] = q[64];
  };
  auto product = [&](const double2 (&b_)[2], auto G, auto J) {  // two terms of group g
    constexpr int g = decltype(G)::value, j = decltype(J)::value, pi = (4 * g + j) & 15;
    pr[g & 1][2 * j] = av[g & 1][j].x * row_bcast<pi>(b_[g / 4].x);
    pr[g & 1][2 * j + 1] = av[g & 1][j].y * row_bcast<pi>(b_[g / 4].y);
  };
  // add group g; next: forms the two terms j of the group after it between
  // the additions
  auto add = [&](auto G, auto next) {
    constexpr int g = decltype(G)::value;
    unroll<0, 4>([&](auto J) {
      constexpr int j = decltype(J)::value;
      next(J);
      acc = acc + pr[g & 1][2 * j];
      acc = acc + pr[g & 1][2 * j + 1];
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  constexpr std::integral_constant<int, 0> g0{};
  constexpr std::integral_constant<int, 1> g1{};
  bar_reader();  // chunk 0 has landed
  read_b(0, bv);
  read_a(0, g0);
  read_a(0, g1);
  unroll<0, 4>([&](auto J) { product(bv, g0, J); });
  int sl = 0;
  for (int c = 0; c < nlast; ++c) {
    const int sn = sl + 1 == R ? 0 : sl + 1;
    unroll<0, 8>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if constexpr (g == 4) bar_reader();
      if constexpr (g == 5) read_b(sn, bn);
      read_a(g + 2 < 8 ? sl : sn, std::integral_constant<int, (g + 2) & 7>{});
      add(G, [&](auto J) {
        if constexpr (g < 7) product(bv, std::integral_constant<int, (g + 1) & 7>{}, J);
        else product(bn, g0, J);
      });
    });
    bv[0] = bn[0];
    bv[1] = bn[1];
    sl = sn;
  }
  const int kc = K - nlast * GS_K;
  unroll<0, 8>([&](auto G) {
    constexpr int g = decltype(G)::value;
    if (8 * g < kc) {
      if constexpr (g + 2 < 8) read_a(sl, std::integral_constant<int, (g + 2) & 7>{});
      add(G, [&](auto J) {
        if constexpr (g < 7) product(bv, std::integral_constant<int, (g + 1) & 7>{}, J);
      });
    }
  });
  // through LDS to the epilogue's order, consecutive columns adjacent
  Ts[lane & 15][4 * wave + (lane >> 4)] = acc;
  __syncthreads();
  if (eok) {
    const double d = Ts[t / NT][t % NT];
    switch (p.ep) {
      case EP_FWD:
        p.dum0[(long)em * p.dum0_stride + en] = xv;
        *ex = xv - d;
        break;
      case EP_BWD:
        *ex = xv + d;
        p.out[(long)em * p.out_ld + en] = d;
        if (p.g) p.g[(long)em * p.out_ld + en] = d * (double)cyv;
        break;
      default:  // EP_CPL
        p.out[(long)em * p.out_ld + en] = d;
        break;
    }
  }
  span_end(p.tspan);
}

// The same products for few right-hand sides (M <= MR <= 8), where the kernel
// above leaves most of its 16-row lanes idle and a launch lasts as long as
// one sum: the products of a term are formed apart from the additions.  Two
// wavefronts form them (a half wavefront takes one of the tile's four columns
// and 64 k at a time, the loads of both operands R chunks ahead in
// registers) and leave them in LDS; the third only adds, one sum a lane, at
// the rate of an addition and its LDS read instead of the multiply's, the
// broadcast's and the addition's (10 against 21 clocks a term: one right-hand
// side at 720 columns takes 6.3 us, 9.5 in the kernel above, 17.4 before
// both).  Products past K are +0, which keeps the bits of a sum that started
// from +0.  Barriers as above: one a chunk, in the middle of its sum, with
// three chunks in LDS.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // at any 8-byte boundary

template <int MR, int R>
__global__ __launch_bounds__(192) void gemm_seq_few_kernel(GemmArgs p) {
  __shared__ __align__(16) double P[3][4 * MR][GS_K + 2];
  span_begin(p.tspan);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n0 = 4 * blockIdx.x, K = p.K;
  const int nlast = (K + GS_K - 1) / GS_K - 1;
  if (wave > 0) {
    const int col = 2 * (wave - 1) + (lane >> 5), kp = 2 * (lane & 31);
    const double *bcol = p.b + (long)min(n0 + col, p.N - 1) * p.b_sn;
    d2u ra[R][MR], rb[R];
    // a chunk past the last loads the last again: the waits count loads
    auto fetch = [&](int c, d2u (&a_)[MR], d2u &b_) {
      const int k = min(min(c, nlast) * GS_K + kp, K - 2);
      b_ = *reinterpret_cast<const d2u *>(bcol + k);
#pragma unroll
      for (int m = 0; m < MR; ++m)
        a_[m] = *reinterpret_cast<const d2u *>(p.a + (long)min(m, p.M - 1) * p.a_sm + k);
    };
#pragma unroll
    for (int d = 0; d < R; ++d) fetch(d, ra[d], rb[d]);
    int buf = 0;
    for (int c0 = 0; c0 <= nlast; c0 += R) {
      unroll<0, R>([&](auto D) {
        constexpr int d = decltype(D)::value;
        const int c = c0 + d;
        if (c <= nlast) {
          // past the end the pair came from K - 2: its second product is k = K - 1's
          const int sh = c * GS_K + kp - (K - 2);
#pragma unroll
          for (int m = 0; m < MR; ++m) {
            const double q0 = ra[d][m].x * rb[d].x, q1 = ra[d][m].y * rb[d].y;
            *reinterpret_cast<double2 *>(&P[buf][4 * m + col][kp]) =
                make_double2(sh <= 0 ? q0 : (sh == 1 ? q1 : 0.0), sh <= 0 ? q1 : 0.0);
          }
          fetch(c + R, ra[d], rb[d]);
          bar_written();
          buf = buf == 2 ? 0 : buf + 1;
        }
      });
    }
    if (p.tspan) __syncthreads();  // span_end's of the adding wavefront
    return;
  }
  const int m = min(lane >> 2, p.M - 1), n = min(n0 + (lane & 3), p.N - 1);
  const bool ok = (lane >> 2) < p.M && n0 + (lane & 3) < p.N;
  double xv = 0.0;
  float cyv = 0.f;
  double *ex = nullptr;
  if (p.ep != EP_CPL) {
    ex = p.x + (long)m * p.x_stride + f2(p.i2 + 2, n + 2, p.xrow);
    xv = *ex;
    if (p.g) cyv = p.cy[(long)n + (long)(p.cyrow - 1) * p.i2];
  }
  const double *pl = &P[0][min(lane, 4 * MR - 1)][0];
  constexpr int PB = sizeof(P[0]) / sizeof(double);
  double acc = 0.0;
  double2 v[4][4];
  auto read = [&](const double *q, auto G) {
    constexpr int g = decltype(G)::value;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[g & 3][j] = *reinterpret_cast<const double2 *>(q + 8 * g + 2 * j);
  };
  auto add = [&](auto G, auto then) {  // then: the read into the slots this group leaves
    constexpr int g = decltype(G)::value;
    double2 w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = v[g & 3][j];
    then();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc = acc + w[j].x;
      acc = acc + w[j].y;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // groups of 8 k, requested four groups ahead (an LDS read takes as long as
  // two or three groups' additions); the second half of a chunk requests the
  // next one's first half
  const double *q = pl;
  int buf = 0;
  bar_reader();
  unroll<0, 4>([&](auto G) { read(q, G); });
  for (int c = 0; c < nlast; ++c) {
    buf = buf == 2 ? 0 : buf + 1;
    const double *qn = pl + buf * PB;
    unroll<0, 8>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if constexpr (g == 4) bar_reader();
      add(G, [&] { read(g < 4 ? q : qn, std::integral_constant<int, (g + 4) & 7>{}); });
    });
    q = qn;
  }
  const int kc = K - nlast * GS_K;
  unroll<0, 8>([&](auto G) {
    constexpr int g = decltype(G)::value;
    if (8 * g < kc)
      add(G, [&] {
        if constexpr (g < 4) read(q, std::integral_constant<int, (g + 4) & 7>{});
      });
  });
  if (ok) {
    switch (p.ep) {
      case EP_FWD:
        p.dum0[(long)m * p.dum0_stride + n] = xv;
        *ex = xv - acc;
        break;
      case EP_BWD:
        *ex = xv + acc;
        p.out[(long)m * p.out_ld + n] = acc;
        if (p.g) p.g[(long)m * p.out_ld + n] = acc * (double)cyv;
        break;
      default:  // EP_CPL
        p.out[(long)m * p.out_ld + n] = acc;
        break;
    }
  }
  span_end(p.tspan);
}

// Square products of the influence build, D = A B, or 0 - A B by successive
// subtractions (neg): n x n column-major matrices, so A and D have consecutive m
// adjacent and B consecutive k.  One output per thread, tile 16 (m) x 16 (n), K in
// chunks of 64 staged through LDS.
constexpr int GT_M = 16, GT_N = 16, GT_K = 64;

__global__ __launch_bounds__(256) void gemm_square_kernel(const double *a, const double *b, double *out,
                                                          int n, int neg) {
  // both tiles k-contiguous (rows of GT_K + 2 doubles, 16-byte aligned) so a
  // thread reads two consecutive k of each operand with one 128-bit load
  __shared__ __align__(16) double As[GT_M][GT_K + 2];
  __shared__ __align__(16) double Bs[GT_N][GT_K + 2];
  const int t = threadIdx.x;
  // XCD-aware placement: the row tiles of one column tile read that tile of B
  // from HBM once (the others from the XCD's L2); ids past the last column tile
  // have no tile
  const int ntl = (n + GT_N - 1) / GT_N;
  int tcol, trow;
  if (!tile_of(blockIdx.x, ntl, ntl, tcol, trow)) return;
  const int n0 = tcol * GT_N, m0 = trow * GT_M;
  const int tn = t % GT_N, tm = t / GT_N;
  // staging: each thread moves 4 elements of A (m fastest) and 4 of B (k
  // fastest) per chunk
  double ra[4], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int idx = t + 256 * q;
      const int m = m0 + idx % GT_M, ka = k0 + idx / GT_M;
      ra[q] = (m < n && ka < n) ? a[(long)m + (long)ka * n] : 0.0;
      const int c = n0 + idx / GT_K, kb = k0 + idx % GT_K;
      rb[q] = (c < n && kb < n) ? b[(long)kb + (long)c * n] : 0.0;
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int idx = t + 256 * q;
      As[idx % GT_M][idx / GT_M] = ra[q];
      Bs[idx / GT_K][idx % GT_K] = rb[q];
    }
  };
  double acc = 0.0;
  // chunks are staged in a ring of PF register slots, fetched PF chunks
  // ahead of their use, so the global latency overlaps PF chunks of compute
  constexpr int PF = 3;
  double ra_r[PF][4], rb_r[PF][4];
  const int nchunk = (n + GT_K - 1) / GT_K;
  auto fetch_to = [&](int c, double (&ra_)[4], double (&rb_)[4]) {
    fetch(c * GT_K);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ra_[q] = ra[q];
      rb_[q] = rb[q];
    }
  };
#pragma unroll
  for (int d = 0; d < PF; ++d)
    if (d < nchunk) fetch_to(d, ra_r[d], rb_r[d]);
  for (int c0 = 0; c0 < nchunk; c0 += PF) {
#pragma unroll
    for (int d = 0; d < PF; ++d) {
      const int c = c0 + d;
      if (c >= nchunk) break;
      const int k0 = c * GT_K;
      const int kc = min(GT_K, n - k0);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ra[q] = ra_r[d][q];
        rb[q] = rb_r[d][q];
      }
      stash();
      __syncthreads();
      if (c + PF < nchunk) fetch_to(c + PF, ra_r[d], rb_r[d]);
      const double2 *ar = reinterpret_cast<const double2 *>(&As[tm][0]);
      const double2 *br = reinterpret_cast<const double2 *>(&Bs[tn][0]);
      const int kc2 = kc / 2;
      if (kc == GT_K) {
        // a whole chunk in groups of 16 k: the group's LDS reads are issued
        // one group ahead and its 16 products (independent of the sum) are
        // formed before the 16 dependent additions, which then follow one
        // another at the add latency instead of each waiting for its
        // multiply.  Same products, same order of additions.
        constexpr int GP = 8;  // k pairs per group
        double2 a_c[GP], b_c[GP], a_n[GP], b_n[GP];
#pragma unroll
        for (int j = 0; j < GP; ++j) {
          a_c[j] = ar[j];
          b_c[j] = br[j];
        }
#pragma unroll
        for (int g = 0; g < GT_K / 2 / GP; ++g) {
          if (g + 1 < GT_K / 2 / GP) {
#pragma unroll
            for (int j = 0; j < GP; ++j) {
              a_n[j] = ar[(g + 1) * GP + j];
              b_n[j] = br[(g + 1) * GP + j];
            }
          }
          double pr[2 * GP];
#pragma unroll
          for (int j = 0; j < GP; ++j) {
            pr[2 * j] = a_c[j].x * b_c[j].x;
            pr[2 * j + 1] = a_c[j].y * b_c[j].y;
          }
          if (neg) {
#pragma unroll
            for (int j = 0; j < 2 * GP; ++j) acc = acc - pr[j];
          } else {
#pragma unroll
            for (int j = 0; j < 2 * GP; ++j) acc = acc + pr[j];
          }
#pragma unroll
          for (int j = 0; j < GP; ++j) {
            a_c[j] = a_n[j];
            b_c[j] = b_n[j];
          }
        }
      } else if (neg) {
        for (int k2 = 0; k2 < kc2; ++k2) {
          const double2 av = ar[k2], bv = br[k2];
          acc = acc - av.x * bv.x;
          acc = acc - av.y * bv.y;
        }
        if (kc & 1) acc = acc - As[tm][kc - 1] * Bs[tn][kc - 1];
      } else {
        for (int k2 = 0; k2 < kc2; ++k2) {
          const double2 av = ar[k2], bv = br[k2];
          acc = acc + av.x * bv.x;
          acc = acc + av.y * bv.y;
        }
        if (kc & 1) acc = acc + As[tm][kc - 1] * Bs[tn][kc - 1];
      }
    }
  }
  const int col = n0 + tn, row = m0 + tm;
  if (col < n && row < n) out[(long)row + (long)col * n] = acc;
}

hipError_t launch_square_product(const double *a, const double *b, double *out, int n, bool neg, hipStream_t st) {
  if (n < 1) return hipErrorInvalidValue;
  const int ntl = (n + GT_N - 1) / GT_N;
  hipLaunchKernelGGL(gemm_square_kernel, dim3((unsigned)placed_workgroups(ntl, ntl)), dim3(256), 0, st, a, b, out, n,
                     neg ? 1 : 0);
  return hipGetLastError();
}

// T(i, k) = R(i, k) * CY(k, cyrow): columns of an n x n column-major matrix
// scaled by one row of the north coefficient.
__global__ void scale_cols_kernel(const double *r, const float *cy, int cyrow, int i2, double *t) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long)i2 * i2) return;
  const int k = (int)(q / i2);
  t[q] = r[q] * (double)cy[(long)k + (long)(cyrow - 1) * i2];
}

hipError_t launch_scale_cols(const double *r, const float *cy, int cyrow, int i2, double *t,
                             hipStream_t st) {
  const long n = (long)i2 * i2;
  hipLaunchKernelGGL(scale_cols_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, r, cy,
                     cyrow, i2, t);
  return hipGetLastError();
}

// Computing wavefronts per workgroup of gemm_seq_kernel: as few of 1, 2, 4 and 8
// as leave at most one workgroup per CU, so that no CU runs two workgroups while
// another has none.  That is 240 of the 256 CUs at 960 columns and 64 right-hand
// sides, but 180 at 720 x 32, 720 x 64, 1440 x 32 and 1440 x 64, 152 at 1200 x 64
// and 135 at 1440 x 48 (columns x right-hand sides).
static int gemm_seq_waves(const GemmArgs &a) {
  const long nmb = (a.M + 15) / 16;
  for (int nw : {1, 2, 4})
    if (nmb * ((a.N + 4 * nw - 1) / (4 * nw)) <= 256) return nw;
  return 8;
}
// Right-hand sides up to which the sums are added apart; past 8 the forming
// wavefronts would read more rows than they can keep ahead.  gemm_seq_kernel takes
// the same time for any count up to 16, so 8 against 9 right-hand sides compares
// the two (a pass of 8 blocks): 173 and 177 us at 360 columns, 241 and 262 at 720,
// 272 and 306 at 960, 404 and 421 at 1440, but 150 and 142 at 200, 140 and 131 at
// 130.  One right-hand side: 121 at 200, 191 at 720.
constexpr int GS_FEW = 8;

long gemm_workgroups(const GemmArgs &a) {
  if (a.M <= GS_FEW) return (a.N + 3) / 4;
  const int nt = 4 * gemm_seq_waves(a);
  return 8L * ((a.M + 15) / 16) * (((a.N + nt - 1) / nt + 7) / 8);
}

template <int NW, int NL, int R, int W>
static void gemm_seq_go(const GemmArgs &a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid((unsigned)gemm_workgroups(a)), block(64 * (NW + NL));
  if (ev0) hipExtLaunchKernelGGL((gemm_seq_kernel<NW, NL, R, W>), grid, block, 0, st, ev0, ev1, 0, a);
  else hipLaunchKernelGGL((gemm_seq_kernel<NW, NL, R, W>), grid, block, 0, st, a);
}

template <int MR, int R>
static void gemm_few_go(const GemmArgs &a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid((unsigned)gemm_workgroups(a)), block(192);
  if (ev0) hipExtLaunchKernelGGL((gemm_seq_few_kernel<MR, R>), grid, block, 0, st, ev0, ev1, 0, a);
  else hipLaunchKernelGGL((gemm_seq_few_kernel<MR, R>), grid, block, 0, st, a);
}

hipError_t launch_gemm(const GemmArgs &a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  if (a.M < 1 || a.N < 1 || a.K < 2) return hipErrorInvalidValue;
  if (a.M <= GS_FEW) {
    if (a.M == 1) gemm_few_go<1, 12>(a, st, ev0, ev1);
    else if (a.M == 2) gemm_few_go<2, 8>(a, st, ev0, ev1);
    else if (a.M <= 4) gemm_few_go<4, 8>(a, st, ev0, ev1);
    else gemm_few_go<8, 5>(a, st, ev0, ev1);
    return hipGetLastError();
  }
  const int nw = gemm_seq_waves(a);
  // 16-byte DMAs need every run of k at a 16-byte boundary
  const bool w16 = a.K % 2 == 0 && a.a_sm % 2 == 0 && a.b_sn % 2 == 0 &&
                   ((uintptr_t)a.a & 15) == 0 && ((uintptr_t)a.b & 15) == 0;
  if (w16) {
    if (nw == 1) gemm_seq_go<1, 2, 8, 16>(a, st, ev0, ev1);
    else if (nw == 2) gemm_seq_go<2, 2, 6, 16>(a, st, ev0, ev1);
    else if (nw == 4) gemm_seq_go<4, 2, 6, 16>(a, st, ev0, ev1);
    else gemm_seq_go<8, 2, 6, 16>(a, st, ev0, ev1);
  } else {
    if (nw == 1) gemm_seq_go<1, 4, 8, 4>(a, st, ev0, ev1);
    else if (nw == 2) gemm_seq_go<2, 4, 6, 4>(a, st, ev0, ev1);
    else if (nw == 4) gemm_seq_go<4, 4, 6, 4>(a, st, ev0, ev1);
    else gemm_seq_go<8, 8, 6, 4>(a, st, ev0, ev1);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MATINV in LDS for n <= MATINV_LDS_MAX, one workgroup per matrix.
constexpr int MATINV_LDS_MAX = 128;

__global__ __launch_bounds__(256) void matinv_lds_kernel(double *mats, long stride, int n, int *zp) {
  extern __shared__ double sm[];
  double *B = sm;                 // n*n, column-major
  double *b1 = sm + (long)n * n;  // n
  __shared__ double piv;
  __shared__ int zcount;
  double *g = mats + (long)blockIdx.x * stride;
  const int t = threadIdx.x, nt = blockDim.x;
  const int nn = n * n;
  for (int i = t; i < nn; i += nt) B[i] = g[i];
  if (t == 0) zcount = 0;
  __syncthreads();
#define BM(i, j) B[((i) - 1) + ((j) - 1) * n]
  for (int i = 1; i <= n - 1; ++i) {
    if (t == 0) {
      if (BM(i, i) == 0.0) ++zcount;
      piv = 1.0 / BM(i, i);
      BM(i, i) = 1.0;
    }
    __syncthreads();
    const double bp = piv;
    for (int j = 1 + t; j <= n; j += nt) BM(i, j) = BM(i, j) * bp;
    for (int ia = i + 1 + t; ia <= n; ia += nt) b1[ia - 1] = BM(ia, i);
    __syncthreads();
    // rows ia > i: column i is zeroed then updated like every other column
    const int rows = n - i;
    for (int idx = t; idx < rows * n; idx += nt) {
      const int ia = i + 1 + idx % rows, j = 1 + idx / rows;
      const double cur = (j == i) ? 0.0 : BM(ia, j);
      BM(ia, j) = cur - b1[ia - 1] * BM(i, j);
    }
    __syncthreads();
  }
  if (t == 0) {
    if (BM(n, n) == 0.0) ++zcount;
    piv = 1.0 / BM(n, n);
    BM(n, n) = 1.0;
  }
  __syncthreads();
  {
    const double bp = piv;
    for (int j = 1 + t; j <= n; j += nt) BM(n, j) = BM(n, j) * bp;
  }
  __syncthreads();
  for (int i = 2; i <= n; ++i) {
    for (int ib = 1 + t; ib <= i - 1; ib += nt) b1[ib - 1] = BM(ib, i);
    __syncthreads();
    const int rows = i - 1;
    for (int idx = t; idx < rows * n; idx += nt) {
      const int ib = 1 + idx % rows, j = 1 + idx / rows;
      const double cur = (j == i) ? 0.0 : BM(ib, j);
      BM(ib, j) = cur - b1[ib - 1] * BM(i, j);
    }
    __syncthreads();
  }
#undef BM
  for (int i = t; i < nn; i += nt) g[i] = B[i];
  if (t == 0 && zp && zcount) atomicAdd(zp, zcount);
}

bool matinv_uses_lds(int n) {
  return n <= MATINV_LDS_MAX && sizeof(double) * ((size_t)n * n + n) <= 64 * 1024;
}

// LDS-resident elimination when the matrix fits, else the blocked form
// (sevp_matinv.hip) with `scratch` of matinv_blocked_scratch(n, count) doubles.
hipError_t launch_matinv(double *mats, long stride, int n, int count, int *zp, double *scratch,
                         hipStream_t st) {
  if (matinv_uses_lds(n)) {
    const size_t lds = sizeof(double) * ((size_t)n * n + n);
    hipLaunchKernelGGL(matinv_lds_kernel, dim3(count), dim3(256), lds, st, mats, stride, n, zp);
    return hipGetLastError();
  }
  if (!scratch) return hipErrorInvalidValue;
  return launch_matinv_blocked(mats, stride, n, count, zp, scratch, st);
}

// Periodic halo columns at the end of REP1 (MAIN/template/GLOBAL/src/sevp.f90:103-106).
__global__ void halo_fix_kernel(double *x, long xs, int i2, int j2, int nrhs) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)nrhs * j2) return;
  const int r = (int)(t / j2), j = (int)(t % j2) + 2;
  const int i0 = i2 + 2;
  double *xr = x + (long)r * xs;
  xr[f2(i0, 1, j)] = xr[f2(i0, i0 - 1, j)];
  xr[f2(i0, i0, j)] = xr[f2(i0, 2, j)];
}

hipError_t launch_halo_fix(double *x, long xs, int i2, int j2, int nrhs, hipStream_t st) {
  const long n = (long)nrhs * j2;
  hipLaunchKernelGGL(halo_fix_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, xs, i2, j2, nrhs);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Grouped launches of the mixed pass: one launch runs the same step of many
// independent problems (group_entry finds a workgroup's problem), each entry
// with exactly the workgroups and arguments of its own launch, so every value
// written is the one the problem's own launch writes.
template <int K>
__global__ __launch_bounds__(64) void batch_march_kernel(const MarchEnt *__restrict__ tab,
                                                         const int *__restrict__ start, int n) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  const MarchEnt &t = tab[e];
  const int l = b - start[e];
  march_body<K, MODE_PART>(t.m, l % t.ntiles, l / t.ntiles, 0, 1, threadIdx.x);
}

template <int K>
__global__ __launch_bounds__(64) void batch_hom_resid_kernel(const HomResidEnt *__restrict__ tab,
                                                             const int *__restrict__ start, int n) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  const HomResidEnt &t = tab[e];
  hom_resid_body<K>(t.m, t.r, t.ntiles, t.has_resid, b - start[e]);
}

__global__ __launch_bounds__(256) void batch_resid_kernel(const ResidArgs *__restrict__ tab,
                                                          const int *__restrict__ start, int n) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  resid_body(tab[e], (long)(b - start[e]) * 256 + threadIdx.x);
}

// Zero fill of n 32-bit words per entry (the correction arrays of a pass).
__global__ __launch_bounds__(256) void batch_fill_kernel(const FillEnt *__restrict__ tab,
                                                         const int *__restrict__ start, int n) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  const long t = (long)(b - start[e]) * 256 + threadIdx.x;
  if (t < tab[e].n) tab[e].p[t] = 0u;
}

// X += D over the interior of entries whose problem is still refining
// (act[problem] != 0, or every entry when act is null), then, in a second
// launch, the periodic halo columns.
__global__ __launch_bounds__(256) void batch_axpy_kernel(const AxpyEnt *__restrict__ tab,
                                                         const int *__restrict__ start, int n,
                                                         const int *__restrict__ act) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  const AxpyEnt &a = tab[e];
  if (act && !act[a.problem]) return;
  const long t = (long)(b - start[e]) * 256 + threadIdx.x;
  const long np = (long)a.i2 * a.j2;
  if (t >= np * a.nrhs) return;
  const int r = (int)(t / np);
  const long q = t % np;
  const int i = (int)(q % a.i2) + 2, j = (int)(q / a.i2) + 2;
  const long o = f2(a.i2 + 2, i, j);
  a.x[(long)r * a.x_stride + o] += a.d[(long)r * a.d_stride + o];
}

__global__ __launch_bounds__(256) void batch_halo_kernel(const AxpyEnt *__restrict__ tab,
                                                         const int *__restrict__ start, int n,
                                                         const int *__restrict__ act) {
  const int b = blockIdx.x;
  const int e = group_entry(start, n, b);
  const AxpyEnt &a = tab[e];
  if (act && !act[a.problem]) return;
  const long t = (long)(b - start[e]) * 256 + threadIdx.x;
  if (t >= (long)a.nrhs * a.j2) return;
  const int r = (int)(t / a.j2), j = (int)(t % a.j2) + 2;
  const int i0 = a.i2 + 2;
  double *xr = a.x + (long)r * a.x_stride;
  xr[f2(i0, 1, j)] = xr[f2(i0, i0 - 1, j)];
  xr[f2(i0, i0, j)] = xr[f2(i0, 2, j)];
}

static bool batch_grid_ok(int n, long nwg) { return n >= 1 && nwg >= 1 && nwg <= 0x7fffffffL; }

hipError_t launch_batch_march(int K, const MarchEnt *tab, const int *start, int n, long nwg,
                              hipStream_t st) {
  if (!batch_grid_ok(n, nwg)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nwg);
  if (K == 1) hipLaunchKernelGGL((batch_march_kernel<1>), grid, dim3(64), 0, st, tab, start, n);
  else if (K == 2) hipLaunchKernelGGL((batch_march_kernel<2>), grid, dim3(64), 0, st, tab, start, n);
  else if (K == 4) hipLaunchKernelGGL((batch_march_kernel<4>), grid, dim3(64), 0, st, tab, start, n);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_batch_hom_resid(int K, const HomResidEnt *tab, const int *start, int n, long nwg,
                                  hipStream_t st) {
  if (!batch_grid_ok(n, nwg)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nwg);
  if (K == 1) hipLaunchKernelGGL((batch_hom_resid_kernel<1>), grid, dim3(64), 0, st, tab, start, n);
  else if (K == 2) hipLaunchKernelGGL((batch_hom_resid_kernel<2>), grid, dim3(64), 0, st, tab, start, n);
  else if (K == 4) hipLaunchKernelGGL((batch_hom_resid_kernel<4>), grid, dim3(64), 0, st, tab, start, n);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_batch_resid(const ResidArgs *tab, const int *start, int n, long nwg, hipStream_t st) {
  if (!batch_grid_ok(n, nwg)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(batch_resid_kernel, dim3((unsigned)nwg), dim3(256), 0, st, tab, start, n);
  return hipGetLastError();
}

hipError_t launch_batch_fill(const FillEnt *tab, const int *start, int n, long nwg, hipStream_t st) {
  if (!batch_grid_ok(n, nwg)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(batch_fill_kernel, dim3((unsigned)nwg), dim3(256), 0, st, tab, start, n);
  return hipGetLastError();
}

hipError_t launch_batch_axpy(const AxpyEnt *tab, const int *start, int n, long nwg, const int *act,
                             bool halo, hipStream_t st) {
  if (!batch_grid_ok(n, nwg)) return hipErrorInvalidValue;
  if (halo) hipLaunchKernelGGL(batch_halo_kernel, dim3((unsigned)nwg), dim3(256), 0, st, tab, start, n, act);
  else hipLaunchKernelGGL(batch_axpy_kernel, dim3((unsigned)nwg), dim3(256), 0, st, tab, start, n, act);
  return hipGetLastError();
}

}  // namespace sevp

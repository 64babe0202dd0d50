// One launch per block step: the correction product of a full-width SEVP
// pass fused with what depends on it, for the MFMA corrections (FP32 or BF16
// with FP64 refinement, or FP64).
//
// The split-K pass (sevp_mixed.hip) takes four launches per block and writes
// every product as slice partials that the next launch adds up.  Here a
// workgroup computes whole dot products: its W wavefronts split K, each keeps
// one or two 16 x 16 accumulators of the MFMA instruction (two 16-row tiles
// share the matrix operand), and the W partial tiles are added in FP64 in
// wavefront order through LDS, so every output is one fixed sum.  The
// epilogue then does the work that depends only on that output's column:
//
//   forward, block b:  d = e_b RINV1_b.  Block b+1's first march row uses the
//     corrected south row X(IE(b)) - d (never written back: the backward pass
//     restores the uncorrected value anyway, REP1's DUM0), its closure
//     residual e_(b+1) needs the marched rows at the neighbouring columns, so
//     a tile computes 16 columns of d and marches them with DPP row shifts
//     (16 lanes = 16 columns of one right-hand side).  The first row
//     operation takes the free row's neighbours from memory and is exact in
//     every lane; each later one (march rows, then the closure) loses a lane
//     per side, so a tile writes the 16 - 2*steps columns that stay exact
//     (the trapezoid of the march kernels; recomputed columns repeat the
//     same operations on the same operands, so they agree bitwise with the
//     tile that owns them).
//   backward, block b: [c | cpl] = e_b [RINV_b | W_b].  X(JS+1) += c and the
//     closure residual of block b-1, which reads that row only at its own
//     column, are done at once; c and cpl are stored for the homogeneous
//     march of block b, which needs c at the neighbouring columns and runs in
//     the next launch (its workgroups come first), when every column is
//     complete.
//
// Where that saves time (warms) the last workgroups of a launch read the next
// launch's matrices into L2: a launch is a chain of latencies (operands, product,
// epilogue) with the memory idle for most of it.
//
// A pass is 2*NB0 + 1 launches instead of 4*NB0 + 2, each influence matrix is
// read from HBM once for all right-hand sides, and no partial products go
// through memory.  Both operands are in lane tiles, so a wavefront's operand
// for 16 rows (or columns) and 16 k is one contiguous 1 KiB (FP32) run; every
// load address is clamped in bounds instead of masked, so a wavefront issues
// all its loads of a K range before its first wait.  The workgroups of one
// column tile are placed on the same XCD so the tile's matrix columns are
// fetched from HBM once.
#include <hip/hip_ext.h>

#include <type_traits>

#include "sevp_dev.h"
#include "sevp_internal.h"
#include "sevp_march.h"
#include "sevp_tiles.h"

namespace sevp {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// Lane i of each 16-lane row receives lane i-1's (row_shr:1) or lane i+1's
// (row_shl:1) value; the row's edge lane keeps its own.  The edge lanes are
// trapezoid halo columns whose results are never stored.
__device__ __forceinline__ double row_shr1(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x111, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0x111, 0xf, 0xf, false));
}
__device__ __forceinline__ double row_shl1(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x101, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0x101, 0xf, 0xf, false));
}

// BF16 bits of a float, rounded to nearest even (NaN stays a quiet NaN).
__device__ __forceinline__ short bf16_rne(float f) {
  const unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (short)((u >> 16) | 0x40);
  return (short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// The three product arithmetics.  Per chunk of 16 k a lane holds k = 4q ..
// 4q+3 (q = lane / 16) of its A row and B column: FP32 and FP64 take four
// 16x16x4 MFMA steps (one k each; A and B use the same permutation of k, so
// the product is unchanged); BF16 rounds the FP32 error row to BF16 in
// registers and takes one 16x16x16 step with FP32 accumulation.
struct KF32 {
  typedef float A;
  typedef float B;
  typedef float Acc;
  typedef f32x4 AV;
  typedef f32x4 BV;
  typedef f32x4 CV;
  __device__ static int row(int q, int i) { return 4 * q + i; }
  __device__ static CV mma(AV a, BV b, CV c) {
#pragma unroll
    for (int t = 0; t < 4; ++t) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], c, 0, 0, 0);
    return c;
  }
};
struct KF64 {
  typedef double A;
  typedef double B;
  typedef double Acc;
  typedef f64x4 AV;
  typedef f64x4 BV;
  typedef f64x4 CV;
  __device__ static int row(int q, int i) { return q + 4 * i; }  // the FP64 instruction's D layout
  __device__ static CV mma(AV a, BV b, CV c) {
#pragma unroll
    for (int t = 0; t < 4; ++t) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[t], c, 0, 0, 0);
    return c;
  }
};
struct KB16 {
  typedef float A;            // the error rows stay FP32 in memory
  typedef unsigned short B;   // BF16 bits
  typedef float Acc;
  typedef f32x4 AV;
  typedef s16x4 BV;
  typedef f32x4 CV;
  __device__ static int row(int q, int i) { return 4 * q + i; }
  __device__ static CV mma(AV a, BV b, CV c) {
    const s16x4 ab = {bf16_rne(a[0]), bf16_rne(a[1]), bf16_rne(a[2]), bf16_rne(a[3])};
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ab, b, c, 0, 0, 0);
  }
};

// Two workgroups per CU for the FP32 product with 16 wavefronts and one row
// tile (the mixed precision default): at most 64 VGPRs (8 waves per SIMD),
// which the kernels reach without spills when their load groups are halved
// (3 chunks instead of 6: the same loads in flight per CU).  A backward
// launch of two 32-RHS row tiles has about 400 workgroups, more than one per
// CU; with two per CU it runs in one round.  The sums are unchanged.
template <class KT, int W, int MBW>
constexpr bool two_per_cu() {
  return std::is_same<KT, KF32>::value && W == 16 && MBW == 1;
}
template <class KT, int W, int MBW>
constexpr int min_waves_per_simd() {
  return two_per_cu<KT, W, MBW>() ? 8 : 1;
}

// Whether the epilogue's operands come by DMA (see Operands).
template <class KT, int MBW>
constexpr bool operands_by_dma() {
  return std::is_same<KT, KF64>::value && MBW == 1;
}

// Chunks of 16 k per load group: 96 / W, one group at K <= 1536; half that for
// FP64 with two row tiles and for the two-per-CU FP32 kernels.
template <class KT, int W, int MBW>
constexpr int load_group() {
  return ((std::is_same<KT, KF64>::value && MBW == 2) || two_per_cu<KT, W, MBW>()) ? 48 / W : 96 / W;
}
// 1 / d of a group, rounded up.
constexpr int share_of(int group, int d) { return (group + d - 1) / d; }

// Whether there is a kernel in which a wavefront whose share is half or a
// quarter of a group takes that: a load past the share is a repeated one, but a
// compute unit takes 64 bytes a clock either way (one right-hand side, 720
// columns, FP64: 3.52 ms a solve with twelve chunks for each wavefront's six,
// 3.37 without; FP32, 8 wavefronts, 400 columns, 8: 3.26 and 2.77; 800, 24: 8.84
// and 8.30).  Not where the registers are full with the whole group's: FP32 in 16
// wavefronts.
template <class KT, int W, int MBW>
constexpr bool small_groups() {
  return load_group<KT, W, MBW>() == 12 || (load_group<KT, W, MBW>() == 6 && MBW == 1) ||
         std::is_same<KT, KF64>::value;
}

// Partial tile of one wavefront over the chunks [c_lo, c_hi) of 16 k: MBW
// 16-row tiles of A (row tiles mb0 .. mb0+MBW-1, clamped to the last one,
// whose rows are then never stored) times the 16 columns of B around this
// lane's column n.  Chunks are loaded G at a time; a chunk past c_hi loads
// the last one again and is skipped by the MFMA steps (the range is
// wave-uniform), so no load is masked and none waits on another.  PICK: a share
// that half or a quarter of a group holds takes that.
template <class KT, int G, bool PICK, int MBW>
__device__ __forceinline__ void part_tile(const typename KT::A *alt, int mb0, int mtiles,
                                          const typename KT::B *blt, int n, int nchk, int c_lo,
                                          int c_hi, typename KT::CV (&acc)[MBW]) {
  typedef typename KT::AV AV;
  typedef typename KT::BV BV;
  const int lane = threadIdx.x & 63, q = lane >> 4;
  const typename KT::B *bb = blt + ((long)(n >> 4) * nchk * 64 + (n & 15) + 16 * q) * 4;
  const typename KT::A *ab[MBW];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) ab[mb] = alt + ((long)min(mb0 + mb, mtiles - 1) * nchk * 64 + lane) * 4;
  const int clast = max(c_hi - 1, 0);
  auto group = [&](auto size, int c0) {
    constexpr int C = decltype(size)::value;
    AV av[C][MBW];
    BV bv[C];
#pragma unroll
    for (int g = 0; g < C; ++g) {
      const long ch = min(c0 + g, clast);
      bv[g] = *reinterpret_cast<const BV *>(bb + ch * 256);
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb) av[g][mb] = *reinterpret_cast<const AV *>(ab[mb] + ch * 256);
    }
    // every load of the group is issued before the first MFMA step, which
    // then waits only for its own chunk (the FP64 operands' group takes too
    // many registers for that: the compiler interleaves them)
    if constexpr (!std::is_same<KT, KF64>::value) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < C; ++g)
      if (c0 + g < c_hi)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb) acc[mb] = KT::mma(av[g][mb], bv[g], acc[mb]);
  };
  if constexpr (PICK) {
    typedef std::integral_constant<int, share_of(G, 2)> Half;
    typedef std::integral_constant<int, share_of(G, 4)> Quarter;
    const int share = c_hi - c_lo;
    if (share <= Quarter::value) return group(Quarter{}, c_lo);
    if (share <= Half::value) return group(Half{}, c_lo);
  }
  typedef std::integral_constant<int, G> Whole;
  // the first group outside the loop: straight-line code, so its loads
  // follow the caller's earlier loads without waiting for them (the FP64
  // operands keep the plain loop, which needs fewer registers)
  int c0 = c_lo;
  if constexpr (!std::is_same<KT, KF64>::value) {
    group(Whole{}, c0);
    c0 += G;
  }
  for (; c0 < c_hi; c0 += G) group(Whole{}, c0);
}

// The product tile of a workgroup: W wavefronts, each its share of the K
// chunks; their partial tiles go to LDS and thread t < 256 MBW receives the FP64
// sum over the wavefronts, in wavefront order, of row t / 16 (of the MBW row
// tiles) and column t % 16 of the tile.  Every thread of the workgroup must call
// it.
template <class KT, int W, int MBW, bool PICK>
__device__ __forceinline__ double product_tile(const typename KT::A *alt, int mb0, int mtiles,
                                               const typename KT::B *blt, int n, int K,
                                               typename KT::Acc *red) {
  const int lane = threadIdx.x & 63, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nchk = (K + 15) >> 4;
  const int c_lo = nchk * wave / W, c_hi = nchk * (wave + 1) / W;
  typename KT::CV acc[MBW];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) acc[mb] = typename KT::CV{0, 0, 0, 0};
  part_tile<KT, load_group<KT, W, MBW>(), PICK, MBW>(alt, mb0, mtiles, blt, n, nchk, c_lo, c_hi, acc);
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[(wave * MBW + mb) * 256 + KT::row(q, i) * 16 + (lane & 15)] = acc[mb][i];
  if constexpr (operands_by_dma<KT, MBW>())
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the epilogue's operands (Operands) too
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x < 256 * MBW)
#pragma unroll
    for (int w = 0; w < W; ++w) s += (double)red[w * 256 * MBW + threadIdx.x];
  return s;
}

// Kernel arguments in scalar registers from here on: loaded together, not one
// part after another behind the branches that lead to their use (with
// workgroup_id, a pass at 200 x 152, FP32, 8 wavefronts, one right-hand side: 663
// us before, 637 with; 720 x 360 FP64, 16: 2250 and 2190).
template <class T, class... More>
__device__ __forceinline__ void have(T v, More... more) {
  asm volatile("" ::"s"(v));
  if constexpr (sizeof...(more) > 0) have(more...);
}
// blockIdx.x in a scalar register: what depends on it are then scalar
// operations and branches.  (Behind span_begin's test of a lane the compiler
// keeps it in a vector register, and masks each of a launch's parts by lanes.)
__device__ __forceinline__ int workgroup_id() {
  int wg = blockIdx.x;
  asm volatile("" : "+s"(wg));
  return wg;
}

// Workgroup wg of the last ones of a launch: the matrix columns that the next
// launch's workgroups of one column tile read (n(tile, i), i = 0..15, of the
// next launch's ntiles), a line a lane, into the L2 of their XCD.  The memory
// is idle for most of a launch, and the next one begins with reading its matrix.
template <class KT, int W, class F>
__device__ __forceinline__ void warm_next(int wg, int ntiles, const void *next, int nchk, F &&n) {
  constexpr int STEP = 128 / (int)sizeof(typename KT::BV);  // columns a line
  constexpr int NS = STEP < 16 ? 16 / STEP + 1 : 2;         // lines that 16 columns may lie in, per q
  constexpr int CPI = 64 / (4 * NS);                        // chunks an instruction
  __shared__ uint32_t into[64];
  int tile;
  if (!warm_tile(wg, ntiles, tile)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int q = lane & 3, k = (lane >> 2) % NS, sub = lane / (4 * NS);
  const int col = n(tile, min(k * STEP, 15));
  const typename KT::B *src = static_cast<const typename KT::B *>(next) +
                              ((long)(col >> 4) * nchk * 64 + (col & 15) + 16 * q) * 4;
  for (int i = wave; i * CPI < nchk; i += W) {
    const int ch = i * CPI + sub;
    if (sub < CPI && ch < nchk)
      __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void *)(src + (long)ch * 256),
                                       (__attribute__((address_space(3))) void *)(into), 4, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The right-hand sides of a launch: FP32 (a solve's s) or FP64 (a
// refinement residual), a template parameter so that their loads need no
// branch.
template <class FT>
__device__ __forceinline__ const FT *rhs_ptr(const float *f, const double *f64) {
  if constexpr (std::is_same<FT, double>::value) return f64;
  else return f;
}

// FP64, one row tile: the epilogue's operands that do not depend on the
// product, fetched before it into LDS by DMA, so that they are on their way with
// the product's operands, which take the registers, and there when the product is
// (720 columns, one right-hand side: 3.37 ms a solve with them loaded behind the
// product, 3.16 with these; 800 columns, 24: 3.83 and 3.71).  FP32 and BF16
// launches are slower with these than with registers (8 wavefronts: 8.51 ms
// against 8.35 at 800 columns) or without (16: 35.9 against 35.2 at 1440 x 720
// with 64), their product's loads waiting behind them in every wavefront; so are
// FP64 launches of two row tiles, where the same wavefronts share twice the DMAs
// out (a pass with 24 right-hand sides at 64 x 48, 8 wavefronts: 230 us against
// 205; 16: 889 against 858 at 200 x 152, 3390 against 3270 at 720 x 360).
//
// Output t of the workgroup has dword k at op[k][t]; the wavefronts share the
// dwords out (those of 256 outputs each, every NS-th), all at the addresses
// of output threadIdx.x % 256, so an address is valid for every thread.
template <int W, int N>
struct Operands {
  static constexpr int T = 256, NS = W / 4;
  uint32_t *op;  // N * T dwords
  template <int K>
  __device__ void dma(const void *src, int part) const {
    if (K % NS == part)
      __builtin_amdgcn_global_load_lds(
          (__attribute__((address_space(1))) void *)(src),
          (__attribute__((address_space(3))) void *)(op + K * T +
                                                     __builtin_amdgcn_readfirstlane(threadIdx.x & (T - 64))),
          4, 0, 0);
  }
  // dword K, dwords K and K + 1: a value's own address
  template <int K>
  __device__ void fetch(const float *src, int part) const { dma<K>(src, part); }
  template <int K>
  __device__ void fetch(const double *src, int part) const {
    dma<K>(src, part);
    dma<K + 1>(reinterpret_cast<const char *>(src) + 4, part);
  }
  // f(part) for the wavefront's part, a constant in each copy of f's code
  template <class F>
  __device__ static void share(F &&f) {
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    unroll<0, NS>([&](auto P) {
      if (part == decltype(P)::value) f(P);
    });
  }
  __device__ float f32(int k) const { return __uint_as_float(op[k * T + threadIdx.x]); }
  __device__ double f64(int k) const {
    return __hiloint2double((int)op[(k + 1) * T + threadIdx.x], (int)op[k * T + threadIdx.x]);
  }
  template <class V>
  __device__ V value(int k) const {
    if constexpr (std::is_same<V, double>::value) return f64(k);
    else return f32(k);
  }
};

// ------------------------------------------------------------------ forward
// Output t of a forward workgroup: right-hand side m (mm: 0 past the last) and
// tile column col.
struct FwdCol {
  int col, m, mm, c, pc, xc, xcw, xce;
  bool halo;
  // T: outputs per workgroup (a thread past them reads right-hand side 0)
  __device__ __forceinline__ FwdCol(const FusedFwdArgs &p, int tile, int mb0, int t, int T) {
    const int i2 = p.i2, i0 = i2 + 2;
    col = t & 15;
    m = 16 * mb0 + (t >> 4);
    mm = t < T && m < p.M ? m : 0;
    // interior column (1-based, before wrapping) of this lane's tile column
    c = fused_fwd_column(tile, p.steps, col);
    pc = fused_fwd_matrix_column(c, i2, p.periodic);
    halo = false;
    if (p.periodic) {
      // X columns of the west and east neighbours (wrapped, or the Dirichlet
      // column at the edge)
      xcw = (pc == 1 ? i2 : pc - 1) + 1;
      xce = (pc == i2 ? 1 : pc + 1) + 1;
    } else {
      halo = c < 1 || c > i2;  // Dirichlet columns: X holds the boundary values
      xcw = max(min(c - 1, i2 + 1), 0) + 1;
      xce = max(min(c + 1, i2 + 1), 0) + 1;
    }
    xc = halo ? (c < 1 ? 1 : i0) : pc + 1;  // X column
  }
};

// The epilogue operands that do not depend on the product are X(., JS),
// X(., JS+1) with its west and east neighbours, X(., IE+1), and the coefficients
// and right-hand side of the first march row and of the closure row.  They are
// requested before it, from addresses valid for every thread (threads without
// an output read right-hand side 0), so no load is predicated and the product's
// loads are issued without waiting for them: all of them by DMA in FP64 with one
// row tile; the X values into registers otherwise, and with 8 wavefronts of FP32 or
// BF16 the others too (16 wavefronts leave no registers for them, nor do the FP64
// operands).
template <class KT, int W, int MBW, bool PICK, bool WARM, class FT>
__global__ __launch_bounds__(64 * W, (min_waves_per_simd<KT, W, MBW>())) void fused_fwd_kernel(FusedFwdArgs p) {
  constexpr int kVs = 0, kVc = 2, kFw = 4, kFe = 6, kNorth = 8, kRow1 = 10, kRowR = 15, kF1 = 20,
                kFr = 20 + sizeof(FT) / 4, kN = 20 + sizeof(FT) / 2;
  __shared__ typename KT::Acc red[W * 256 * MBW];
  constexpr bool DM = operands_by_dma<KT, MBW>(), PF = !std::is_same<KT, KF64>::value && W == 8;
  __shared__ uint32_t opmem[DM ? kN * 256 : 1];
  const Operands<W, kN> ops{opmem};
  const int wg = workgroup_id();
  have(p.ntiles, p.nmb, p.nprod, p.a, p.b, p.M, p.i2, p.periodic, p.js, p.jf, p.ieb, p.steps, p.x, p.x_stride);
  have(p.ax, p.ay, p.bb, p.cx, p.cy, rhs_ptr<FT>(p.f, p.f64), p.f_stride);
  span_begin(p.tspan);
  int tile, mbg;
  if (WARM && __builtin_expect(wg >= p.nprod, 0)) {
    warm_next<KT, W>(wg - p.nprod, p.next_tiles, p.next, (p.i2 + 15) >> 4, [&](int tl, int i) {
      return fused_fwd_matrix_column(fused_fwd_column(tl, p.next_steps, i), p.i2, p.periodic) - 1;
    });
  } else if (tile_of(wg, p.ntiles, p.nmb, tile, mbg)) {
    const int steps = p.steps;
    const int i2 = p.i2, i0 = i2 + 2, nchk = (i2 + 15) >> 4;
    const int js = p.js, jf = p.jf, ieb = p.ieb;
    const int jr = ieb - 1;                  // closure row
    const int j1 = steps > 0 ? js : jr;     // first march row (a valid row either way)
    const int tid = DM ? threadIdx.x & 255 : threadIdx.x;
    int pcol;
    double vs, vc, fw, fe, xnorth;
    FT f1, fr;
    float c1[5], cr[5];
    // the free row's neighbours come from memory (that row is not written
    // in the forward pass), so the first row operation is exact in every
    // lane and each later one loses one lane per side
    {
      const FwdCol o(p, tile, MBW * mbg, tid, 256 * MBW);
      pcol = o.pc - 1;
      const double *x = p.x + (long)o.mm * p.x_stride;
      const FT *f = rhs_ptr<FT>(p.f, p.f64) + (long)o.mm * p.f_stride;
      const long o1 = pcol + (long)(j1 - 1) * i2, orr = pcol + (long)(jr - 1) * i2;
      const float *const cfs[5] = {p.ax, p.ay, p.bb, p.cx, p.cy};
      if constexpr (DM) {
        ops.share([&](auto part) {
          ops.template fetch<kVs>(x + f2(i0, o.xc, js), part);
          ops.template fetch<kVc>(x + f2(i0, o.xc, js + 1), part);
          ops.template fetch<kFw>(x + f2(i0, o.xcw, js + 1), part);
          ops.template fetch<kFe>(x + f2(i0, o.xce, js + 1), part);
          ops.template fetch<kNorth>(x + f2(i0, o.xc, ieb + 1), part);
          unroll<0, 5>([&](auto I) {
            constexpr int i = decltype(I)::value;
            ops.template fetch<kRow1 + i>(cfs[i] + o1, part);
            ops.template fetch<kRowR + i>(cfs[i] + orr, part);
          });
          ops.template fetch<kF1>(f + o1, part);
          ops.template fetch<kFr>(f + orr, part);
        });
      } else {
        vs = x[f2(i0, o.xc, js)];
        vc = x[f2(i0, o.xc, js + 1)];
        fw = x[f2(i0, o.xcw, js + 1)];
        fe = x[f2(i0, o.xce, js + 1)];
        xnorth = x[f2(i0, o.xc, ieb + 1)];
        if constexpr (PF) {  // kept in their own precision until used
          f1 = f[o1];
          fr = f[orr];
#pragma unroll
          for (int i = 0; i < 5; ++i) {
            c1[i] = cfs[i][o1];
            cr[i] = cfs[i][orr];
          }
        }
      }
    }
    const double d = product_tile<KT, W, MBW, PICK>((const typename KT::A *)p.a, MBW * mbg, (p.M + 15) >> 4,
                                              (const typename KT::B *)p.b, pcol, i2, red);
    int again = tid;
    if constexpr (DM) asm volatile("" : "+v"(again));  // worked out anew rather than kept in registers
    const FwdCol o(p, tile, MBW * mbg, again, 256 * MBW);
    const bool out = o.col >= steps && o.col < 16 - steps && o.c >= 1 && o.c <= i2;
    if (threadIdx.x < 256 * MBW && o.m < p.M) {
      const int m = o.m, pc = o.pc, xc = o.xc;
      const bool halo = o.halo;
      const long co = pc - 1;
      double *x = p.x + (long)m * p.x_stride;
      const FT *f = rhs_ptr<FT>(p.f, p.f64) + (long)m * p.f_stride;
      auto cf = [&](const float *arr, int j) -> double { return (double)arr[co + (long)(j - 1) * i2]; };
      auto fv = [&](int j) -> double { return (double)f[co + (long)(j - 1) * i2]; };
      if constexpr (DM) {
        vs = ops.f64(kVs);
        vc = ops.f64(kVc);
        fw = ops.f64(kFw);
        fe = ops.f64(kFe);
        xnorth = ops.f64(kNorth);
        f1 = ops.template value<FT>(kF1);
        fr = ops.template value<FT>(kFr);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          c1[i] = ops.f32(kRow1 + i);
          cr[i] = ops.f32(kRowR + i);
        }
      } else if constexpr (!PF) {
        const long o1 = co + (long)(j1 - 1) * i2, orr = co + (long)(jr - 1) * i2;
        f1 = f[o1];
        c1[0] = p.ax[o1]; c1[1] = p.ay[o1]; c1[2] = p.bb[o1]; c1[3] = p.cx[o1]; c1[4] = p.cy[o1];
        fr = f[orr];
        cr[0] = p.ax[orr]; cr[1] = p.ay[orr]; cr[2] = p.bb[orr]; cr[3] = p.cx[orr]; cr[4] = p.cy[orr];
      }
      if (!halo) vs = vs - d;  // the south row as block b's correction leaves it
      if (p.d_out && out) p.d_out[(long)m * i2 + pc - 1] = d;
      for (int j = js; j <= jf; ++j) {
        const double sw = row_shr1(vc), se = row_shl1(vc);
        const double xw = j == js ? fw : sw, xe = j == js ? fe : se;
        double r;
        if (j == js)
          r = ((double)f1 - (double)c1[0] * xw - (double)c1[1] * vs - (double)c1[2] * vc - (double)c1[3] * xe) /
              (double)c1[4];
        else
          r = (fv(j) - cf(p.ax, j) * xw - cf(p.ay, j) * vs - cf(p.bb, j) * vc - cf(p.cx, j) * xe) /
              cf(p.cy, j);
        if (halo) r = x[f2(i0, xc, j + 2)];
        if (out) x[f2(i0, xc, j + 2)] = r;
        vs = vc;
        vc = r;
      }
      const double sw = row_shr1(vc), se = row_shl1(vc);
      const double xw = steps == 0 ? fw : sw, xe = steps == 0 ? fe : se;
      const double e = (double)fr - (double)cr[0] * xw - (double)cr[1] * vs - (double)cr[2] * vc -
                       (double)cr[3] * xe - (double)cr[4] * xnorth;
      if (out) {
        const long eo = lt_index(m, (int)co, nchk);
        if (p.e_out) p.e_out[eo] = e;
        if (p.e32_out) p.e32_out[eo] = (float)e;
      }
    }
  }
  span_end(p.tspan);
}

// ----------------------------------------------------------------- backward
// Workgroups [0, nhom_wg): the homogeneous march of block b+1, one wavefront
// per (tile, RHS), first so that the launch's longest dependent chain starts
// at once; then the product tiles of RINV_b (with the epilogue), then, when
// W_b is given, those of W_b (the coupling row, only stored).  The epilogue
// operands (five X values, the right-hand side and coefficients of the closure
// row of block b-1 and the forward correction of its south row) are requested
// where the forward kernel does, from clamped addresses (column I2 for lanes
// past it, row 1 for the closure row of the first block, which has none).
template <class KT, int W, int MBW, bool PICK, bool WARM, class FT>
__global__ __launch_bounds__(64 * W, (min_waves_per_simd<KT, W, MBW>())) void fused_bwd_kernel(FusedBwdArgs p) {
  constexpr int kFree = 0, kSouth = 2, kCen = 4, kW = 6, kE = 8, kDs = 10, kRow = 12, kF = 17,
                kN = 17 + sizeof(FT) / 4;
  __shared__ typename KT::Acc red[W * 256 * MBW];
  constexpr bool DM = operands_by_dma<KT, MBW>(), PF = !std::is_same<KT, KF64>::value && W == 8;
  __shared__ uint32_t opmem[DM ? kN * 256 : 1];
  const Operands<W, kN> ops{opmem};
  const int wg = workgroup_id();
  have(p.nhom_wg, p.ntiles, p.nmb, p.nprod_half, p.a, p.b, p.bw, p.M, p.i2, p.periodic, p.js, p.x, p.x_stride);
  have(p.ax, p.ay, p.bb, p.cx, p.cy, rhs_ptr<FT>(p.f, p.f64), p.f_stride, p.dsouth, p.hfree_out);
  span_begin(p.tspan);
  int tile, mbg;
  if (wg < p.nhom_wg) {
    const long wave = (long)wg * W + (threadIdx.x >> 6);
    if (wave < (long)p.hom_tiles * p.hom.nrhs)
      march_body<1, MODE_HOM>(p.hom, (int)(wave % p.hom_tiles), (int)(wave / p.hom_tiles), 0, 1,
                              threadIdx.x & 63);
  } else {
    const int wp = wg - p.nhom_wg, ww = wp - (p.bw ? 2 : 1) * p.nprod_half;
    if (WARM && __builtin_expect(ww >= 0, 0)) {
      const bool second = ww >= p.nwarm;
      warm_next<KT, W>(second ? ww - p.nwarm : ww, p.ntiles, second ? p.nextw : p.next, (p.i2 + 15) >> 4,
                       [](int tl, int i) { return 16 * tl + i; });
    }
    const bool cpl = wp >= p.nprod_half;
    if ((!WARM || ww < 0) && tile_of(cpl ? wp - p.nprod_half : wp, p.ntiles, p.nmb, tile, mbg)) {
      const int tid = DM ? threadIdx.x & 255 : threadIdx.x;
      const int i2 = p.i2, i0 = i2 + 2, nchk = (i2 + 15) >> 4;
      const int js = p.js, jrow = max(js - 1, 1);
      double xfree, xsouth, xcen, xw, xe, ds;
      FT fr;
      float cr[5];
      // closure row js-1 of block b-1; row js = IE(b-1)
      const double *dsp = p.dsouth ? p.dsouth : p.hfree_out;  // any valid (M, i2) array
      const float *const cfs[5] = {p.ax, p.ay, p.bb, p.cx, p.cy};
      if (!DM || !cpl) {
        const int m = 16 * MBW * mbg + (tid >> 4), mm = tid < 256 * MBW && m < p.M ? m : 0;
        const int cc = min(16 * tile + 1 + (tid & 15), i2);
        const double *x = p.x + (long)mm * p.x_stride;
        const long co = (long)(cc - 1) + (long)(jrow - 1) * i2;  // coefficient row js-1
        const int xcw = p.periodic ? (cc == 1 ? i2 : cc - 1) + 1 : cc;
        const int xce = p.periodic ? (cc == i2 ? 1 : cc + 1) + 1 : cc + 2;
        const FT *fp = rhs_ptr<FT>(p.f, p.f64) + (long)mm * p.f_stride + co;
        const double *dp = dsp + (long)mm * i2 + cc - 1;
        if constexpr (DM) {
          ops.share([&](auto part) {
            ops.template fetch<kFree>(x + f2(i0, cc + 1, js + 1), part);
            ops.template fetch<kSouth>(x + f2(i0, cc + 1, jrow), part);
            ops.template fetch<kCen>(x + f2(i0, cc + 1, js), part);
            ops.template fetch<kW>(x + f2(i0, xcw, js), part);
            ops.template fetch<kE>(x + f2(i0, xce, js), part);
            ops.template fetch<kDs>(dp, part);
            unroll<0, 5>([&](auto I) {
              constexpr int i = decltype(I)::value;
              ops.template fetch<kRow + i>(cfs[i] + co, part);
            });
            ops.template fetch<kF>(fp, part);
          });
        } else {
          xfree = x[f2(i0, cc + 1, js + 1)];
          xsouth = x[f2(i0, cc + 1, jrow)];
          xcen = x[f2(i0, cc + 1, js)];
          xw = x[f2(i0, xcw, js)];
          xe = x[f2(i0, xce, js)];
          if constexpr (PF) {
            fr = *fp;
            ds = *dp;
#pragma unroll
            for (int i = 0; i < 5; ++i) cr[i] = cfs[i][co];
          }
        }
      }
      // lanes past I2 (last tile) read the zero-padded matrix columns
      const double v = product_tile<KT, W, MBW, PICK>((const typename KT::A *)p.a, MBW * mbg, (p.M + 15) >> 4,
                                                (const typename KT::B *)(cpl ? p.bw : p.b), 16 * tile + (tid & 15), i2,
                                                red);
      int again = tid;
      if constexpr (DM) asm volatile("" : "+v"(again));  // as in the forward kernel
      const int m = 16 * MBW * mbg + (again >> 4), c = 16 * tile + 1 + (again & 15);
      if (threadIdx.x < 256 * MBW && m < p.M && c <= i2) {
        const long ro = (long)m * i2 + c - 1;
        if (cpl) {
          p.hcpl_out[ro] = v;
        } else {
          p.hfree_out[ro] = v;
          if constexpr (DM) xfree = ops.f64(kFree);
          const double north = xfree + v;
          p.x[(long)m * p.x_stride + f2(i0, c + 1, js + 1)] = north;
          if (p.do_resid) {
            if constexpr (DM) {
              xsouth = ops.f64(kSouth);
              xcen = ops.f64(kCen);
              xw = ops.f64(kW);
              xe = ops.f64(kE);
              ds = ops.f64(kDs);
              fr = ops.template value<FT>(kF);
#pragma unroll
              for (int i = 0; i < 5; ++i) cr[i] = ops.f32(kRow + i);
            } else if constexpr (!PF) {
              const long co = (long)(c - 1) + (long)(jrow - 1) * i2;
              fr = rhs_ptr<FT>(p.f, p.f64)[(long)m * p.f_stride + co];
              ds = dsp[ro];
#pragma unroll
              for (int i = 0; i < 5; ++i) cr[i] = cfs[i][co];
            }
            if (p.dsouth) xsouth = xsouth - ds;
            const double e = (double)fr - (double)cr[0] * xw - (double)cr[1] * xsouth - (double)cr[2] * xcen -
                             (double)cr[3] * xe - (double)cr[4] * north;
            const long eo = lt_index(m, c - 1, nchk);
            if (p.e_out) p.e_out[eo] = e;
            if (p.e32_out) p.e32_out[eo] = (float)e;
          }
        }
      }
    }
  }
  span_end(p.tspan);
}

// ---------------------------------------------------------------- launchers
// Row tiles per workgroup: the requested 1 or 2 (0: two for FP32 and BF16,
// which share each matrix load, one for FP64), one when M <= 16.  Two row
// tiles halve the matrix reads and the workgroups; FP64 then loads its
// chunks in groups of half the size, within the registers of 16 wavefronts.
static int rows_per_group(int arith, int M, int rows) {
  if (M <= 16) return 1;
  if (rows == 1 || rows == 2) return rows;
  return arith != FUSED_F64 ? 2 : 1;
}

long fused_fwd_workgroups(const FusedFwdArgs &a) {
  return a.nprod + (a.next ? placed_workgroups(a.next_tiles, 1) : 0);
}

long fused_bwd_workgroups(const FusedBwdArgs &a) {
  return a.nhom_wg + (a.bw ? 2L : 1L) * a.nprod_half + (a.next ? 1L : 0L) * a.nwarm + (a.nextw ? 1L : 0L) * a.nwarm;
}

// Whether a launch of wgs product workgroups brings the next one's matrices
// near: while those (two going backward) are about what the L2s hold, 8 of 4 MiB,
// or less, and the chip has room for the workgroups that do it beside the
// product's.  Measured to 33 MB: refined solves, FP64 720 x 360 with one
// right-hand side 3.15 -> 2.38 ms (2.89 by split K), 400 x 190 with one 1.31 ->
// 1.10, 1040 x 500 with 8 5.85 -> 4.84 (5.25 by split K), 800 x 380 with 24 3.71 ->
// 3.33; FP32 800 x 380 with one 7.50 -> 6.79, with 48 (336 workgroups going
// backward) 10.0 -> 9.3, 1200 x 580 with 8 14.6 -> 13.1, with 40 (480) 20.3 -> 20.6.
//
// Where all of a pass's matrices (`set` bytes) stay in the 256 MB last-level
// cache from one pass to the next, they are near enough for wide launches, whose
// workgroups leave no room for more (a pass with and without: FP32 1200 x 24, 196
// MB, 8 right-hand sides 165 and 158 us; 1440 x 28, 232 MB, one 165 and 145; FP64
// 960 x 24, 184 MB, 8 163 and 153; but FP64 1040 x 24, 294 MB, 8 224 and 251, 960 x
// 40, 428 MB, 8 352 and 416).  Narrow ones still gain (FP64 720 x 24, 141 MB, 8 149
// and 154), if they have a kernel to spare for it (warm_go).
static bool warms(int arith, int i2, int waves, int mbw, long set, long wgs) {
  const long n = (i2 + 15) / 16 * 16, elem = arith == FUSED_F64 ? 8 : (arith == FUSED_B16 ? 2 : 4);
  if (2 * n * n * elem > (36L << 20) || wgs > 384) return false;
  if (set > 245000000L) return true;
  return i2 <= 800 && (mbw == 1 || (arith != FUSED_F64 && waves == 8));
}

static int waves_of(int w) { return w == 0 ? FUSED_WAVES : w; }

// Fill the launcher-set fields (tiles, row-tile groups) of the arguments.
int fused_fwd_prepare(FusedFwdArgs &a, int arith) {
  if (a.steps < 0 || 16 - 2 * a.steps < 2 || a.M < 1 || a.M > 64 || a.i2 % 4 != 0) return -1;
  const int w = waves_of(a.waves);
  if (w != 8 && w != 16) return -1;
  if (a.rows < 0 || a.rows > 2) return -1;
  a.ntiles = fused_tiles_fwd(a.i2, a.steps);
  a.mbw = rows_per_group(arith, a.M, a.rows);
  a.nmb = ((a.M + 15) / 16 + a.mbw - 1) / a.mbw;
  a.nprod = (int)placed_workgroups(a.ntiles, a.nmb);
  a.next_tiles = fused_tiles_fwd(a.i2, a.next_steps);
  if (!warms(arith, a.i2, w, a.mbw, a.set, a.nprod)) a.next = nullptr;
  return 0;
}

int fused_bwd_prepare(FusedBwdArgs &a, int arith) {
  if (a.M < 1 || a.M > 64 || a.i2 % 4 != 0) return -1;
  const int w = waves_of(a.waves);
  if (w != 8 && w != 16) return -1;
  if (a.rows < 0 || a.rows > 2) return -1;
  a.ntiles = (a.i2 + 15) / 16;
  a.mbw = rows_per_group(arith, a.M, a.rows);
  a.nmb = ((a.M + 15) / 16 + a.mbw - 1) / a.mbw;
  a.nprod_half = (int)placed_workgroups(a.ntiles, a.nmb);
  a.nwarm = (int)placed_workgroups(a.ntiles, 1);
  if (!warms(arith, a.i2, w, a.mbw, a.set, 2L * a.nprod_half)) a.next = a.nextw = nullptr;
  a.hom_tiles = 0;
  a.nhom_wg = 0;
  if (a.has_hom && a.hom.jf >= a.hom.js) {  // a one-row block has nothing to march
    // one lane per column (any lane width whose tile is positive gives the
    // same values; one keeps the march's registers within the product's)
    a.hom_tiles = march_tiles(a.hom, 1);
    if (a.hom_tiles <= 0) return -1;
    a.nhom_wg = march_workgroups((long)a.hom_tiles * a.hom.nrhs, w);
  }
  return 0;
}

template <class KT, int W, int MBW, bool PICK, bool WARM, class FT>
static void fwd_go(const FusedFwdArgs &a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid((unsigned)fused_fwd_workgroups(a)), block(64 * W);
  if (ev0) hipExtLaunchKernelGGL((fused_fwd_kernel<KT, W, MBW, PICK, WARM, FT>), grid, block, 0, st, ev0, ev1, 0, a);
  else hipLaunchKernelGGL((fused_fwd_kernel<KT, W, MBW, PICK, WARM, FT>), grid, block, 0, st, a);
}

template <class KT, int W, int MBW, bool PICK, bool WARM, class FT>
static void bwd_go(const FusedBwdArgs &a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid((unsigned)fused_bwd_workgroups(a)), block(64 * W);
  if (ev0) hipExtLaunchKernelGGL((fused_bwd_kernel<KT, W, MBW, PICK, WARM, FT>), grid, block, 0, st, ev0, ev1, 0, a);
  else hipLaunchKernelGGL((fused_bwd_kernel<KT, W, MBW, PICK, WARM, FT>), grid, block, 0, st, a);
}

// the right-hand sides' precision -> the kernel that loads them
template <class KT, int W, int MBW, bool PICK, bool WARM>
static void rhs_go(const FusedFwdArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if (a.f64) fwd_go<KT, W, MBW, PICK, WARM, double>(a, st, e0, e1);
  else fwd_go<KT, W, MBW, PICK, WARM, float>(a, st, e0, e1);
}
template <class KT, int W, int MBW, bool PICK, bool WARM>
static void rhs_go(const FusedBwdArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if (a.f64) bwd_go<KT, W, MBW, PICK, WARM, double>(a, st, e0, e1);
  else bwd_go<KT, W, MBW, PICK, WARM, float>(a, st, e0, e1);
}

// The kernel without the part that brings the next matrices near, for launches
// that do not: that part's code alone costs those of two row tiles (a pass with 24
// right-hand sides, 16 wavefronts: FP32 64 x 48 271 us without it, 282 with, 200 x
// 152 929, 977; FP64 800 x 24 224, 234) and the two-per-CU ones, whose registers
// are full (FP32 1440 x 720, 64, two groups: 31.5 ms a solve, 32.2 with).  The
// other kernels take as long either way, or are faster with it (FP32, 8
// wavefronts, two row tiles, 720 x 40: 1.02 of the time without).
template <class KT, int W, int MBW, bool PICK, class Args>
static void warm_go(const Args &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if constexpr (two_per_cu<KT, W, MBW>() || (MBW == 2 && (W == 16 || std::is_same<KT, KF64>::value)))
    if (!a.next) return rhs_go<KT, W, MBW, PICK, false>(a, st, e0, e1);
  rhs_go<KT, W, MBW, PICK, true>(a, st, e0, e1);
}

// The kernel that picks load groups, where most wavefronts' shares are at most
// half of one.  Elsewhere it costs: the choice takes registers and keeps the
// operands requested ahead of the product from staying in flight over it (a pass
// with 8 wavefronts: FP32 1440 x 120, 24 right-hand sides, one row tile 1347 us
// with the choice, 1296 without; FP64 960 x 480, 48, two row tiles 6870, 6640;
// BF16 1200 x 200, 48, one row tile 2260, 2000).  BF16 with few workgroups has
// registers to spare and is faster with it at any width (1200 x 200, one
// right-hand side: 1225, 1329).
template <class KT, int W, int MBW, class Args>
static void go(const Args &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if constexpr (small_groups<KT, W, MBW>()) {
    const int nchk = (a.i2 + 15) / 16, half = share_of(load_group<KT, W, MBW>(), 2);
    if (2 * nchk <= (2 * half + 1) * W || (std::is_same<KT, KB16>::value && a.nmb == 1))
      return warm_go<KT, W, MBW, true>(a, st, e0, e1);
  }
  warm_go<KT, W, MBW, false>(a, st, e0, e1);
}

// (arithmetic, waves, row tiles per workgroup) -> the compiled kernel
template <class Args>
static void dispatch(const Args &a, int arith, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  const bool w16 = waves_of(a.waves) == 16, two = a.mbw == 2;
  if (arith == FUSED_F64) {
    if (w16) two ? go<KF64, 16, 2>(a, st, e0, e1) : go<KF64, 16, 1>(a, st, e0, e1);
    else two ? go<KF64, 8, 2>(a, st, e0, e1) : go<KF64, 8, 1>(a, st, e0, e1);
  } else if (arith == FUSED_B16) {
    if (w16) two ? go<KB16, 16, 2>(a, st, e0, e1) : go<KB16, 16, 1>(a, st, e0, e1);
    else two ? go<KB16, 8, 2>(a, st, e0, e1) : go<KB16, 8, 1>(a, st, e0, e1);
  } else {
    if (w16) two ? go<KF32, 16, 2>(a, st, e0, e1) : go<KF32, 16, 1>(a, st, e0, e1);
    else two ? go<KF32, 8, 2>(a, st, e0, e1) : go<KF32, 8, 1>(a, st, e0, e1);
  }
}

hipError_t launch_fused_fwd(const FusedFwdArgs &a0, int arith, hipStream_t st, hipEvent_t ev0,
                            hipEvent_t ev1) {
  FusedFwdArgs a = a0;
  if (fused_fwd_prepare(a, arith)) return hipErrorInvalidValue;
  dispatch(a, arith, st, ev0, ev1);
  return hipGetLastError();
}

hipError_t launch_fused_bwd(const FusedBwdArgs &a0, int arith, hipStream_t st, hipEvent_t ev0,
                            hipEvent_t ev1) {
  FusedBwdArgs a = a0;
  if (fused_bwd_prepare(a, arith)) return hipErrorInvalidValue;
  dispatch(a, arith, st, ev0, ev1);
  return hipGetLastError();
}

// FP64 column-major (K, N) matrices to BF16 lane tiles (round to nearest
// even via FP32; zero past K or N).
__global__ void cvt_lane_tiles_bf16_kernel(const double *src, unsigned short *dst, int K, int N,
                                           long nmat) {
  const int nchk = (K + 15) / 16;
  const long per = lane_tile_elems(N, K);
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= per * nmat) return;
  const long mat = i / per, r = i % per;
  const int t = (int)(r & 3), l = (int)((r >> 2) & 63);
  const long blk = r >> 8;
  const int ch = (int)(blk % nchk), tile = (int)(blk / nchk);
  const int k = 16 * ch + 4 * (l >> 4) + t, n = 16 * tile + (l & 15);
  dst[i] = (k < K && n < N) ? (unsigned short)bf16_rne((float)src[mat * K * (long)N + k + (long)n * K]) : 0;
}

hipError_t launch_cvt_lane_tiles_bf16(const double *src, unsigned short *dst, int K, int N, long nmat,
                                     hipStream_t st) {
  const long n = lane_tile_elems(N, K) * nmat;
  hipLaunchKernelGGL(cvt_lane_tiles_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     src, dst, K, N, nmat);
  return hipGetLastError();
}

}  // namespace sevp

// Plain FP64 strip SEVP (REPBIR) and the BIR multiplicative strip sweeps.
//
// One workgroup owns one right-hand side and runs the whole chain the
// reference runs on one CPU core: nsweep sweeps x NBIR overlapping strips x
// (forward + backward block march).  The chain is a true data dependency
// (each strip reads the halo columns and interior guess written by the one
// before it, and each block's march starts from the corrected last row of the
// block below), so the only parallelism inside one solve is the strip's
// columns, a lane each in the marching wavefront.  Independent right-hand
// sides run as independent workgroups.
//
// What bounds it is that one wavefront's instructions: it issues one in about
// five clocks whatever it is, a branch in 12 or, taken, 24, a reciprocal in
// 16, so a row step (two wave shifts, four products and the ordered
// differences, a correctly rounded division) is some 55 instructions and a
// closure's dot products some 60, and every wait for memory comes on top.  The
// workgroup's four wavefronts split the work to keep everything else off it:
//  * wave 0, the marcher, reads every row operand from LDS, keeps the live
//    rows in registers, exchanges the stencil's east/west neighbours with DPP
//    wave shifts and writes its results to LDS.  Its only global accesses are
//    the influence-matrix columns (column n of RINV/RINV1 for lane n), loaded
//    into registers a whole block before the closure that uses them.
//  * waves 1-3, the stagers, stream each pass's operands into LDS with
//    global_load_lds DMAs (no registers, no waits while they fly), bring the
//    influence matrices near (into the XCD's L2) and store the march's results
//    back to X and DUM0, each taking every third record.
// A pass is a sequence of records, one per march row or closure, in the order
// the marcher consumes them (the host-built record table, sevp_records.h).
// Records travel in chunks of R through three input buffers: while the
// marcher works on chunk c the stagers fill chunk c+1 and drain chunk c-1,
// and one workgroup barrier ends each chunk on all four wavefronts, so they
// agree on the barrier count by construction (1 + ceil(records / R) per
// pass, plus a pass-end barrier).
//
// A record holds, per column, two quads of dwords and a pair (REC dwords), so
// that the marcher takes it in three reads:
//   quad 0   AX, AY, BB, CX of the row (REAL(4)); of the forward header X(., 1)
//            and X(., 2); of the backward closure's record B X(., JR) and
//            X(., JS+1)
//   quad 1   CY and F of the row (of record B: CY(., JS-1)), then one double:
//            forward march row   the halo, at column 1 X(1, J+1), at column W
//                                X(W+2, J+1)
//            forward closure     the north row X(., IE+1)
//            backward record A   the restored row X(., IE)
//            backward record B   X(., IE+1) of the top block
//            backward march row  the old X(., J+2)
//   pair     a closure's halo.  The marcher leaves its result here (a forward
//            closure's second one, DUM0's row, over quad 0).
// In the 32-lane kernel the pairs are of 64 lanes: the wavefront's idle half
// has somewhere to write.
//
// 720 x 360, 60 strips of 24, blocks of two rows, five sweeps: 58.8 ms for one
// right-hand side, 62.6 for 64 (112 and 123 with a column to a lane, the
// matrices' columns waited for, eight reads a record, three waits on LDS a
// block that the compiler had put before their use; 61 and 81 without the
// stagers' prefetch of the matrices).
//
// Arithmetic follows MAIN/template/GLOBAL/src/sevp.f90:218-328 operation for
// operation (see sevp_dev.h), so results are bitwise equal to the reference.
#include "sevp_dev.h"
#include "sevp_internal.h"

namespace sevp {

// Stager wavefronts per workgroup: a single wavefront's stream of DMAs and
// stores is bound by how many vector memory operations it may have in flight,
// so the records of each chunk are dealt round-robin to NSTG stagers.
constexpr int NSTG = 3;
constexpr int BIR_THREADS = 64 * (1 + NSTG);

template <int WMAX>
struct alignas(16) Stage {
  static constexpr int R = WMAX == 32 ? 24 : 16;  // records per chunk
  static constexpr int NIN = 3;                     // input buffers
  static constexpr int REC = 8 * WMAX + 128;        // dwords per record
  static constexpr int NQ = 4 * WMAX / 64;          // DMAs of a quad
  static constexpr int ND = 2 * WMAX / 64;          // DMAs of the pair
  uint32_t in[NIN][R][REC];
  uint32_t beyond[REC];       // the marcher's prefetch past the last buffer
  double e[WMAX];             // the marcher's residual row, read back as broadcasts
  int desc[4][R][4];          // record-table entries of four chunks
  uint32_t touched[64];       // where the prefetches of influence matrices land
};

// One strip: strip column c (0-based) of the coefficient arrays is physical
// column col(c); X(i, j) = xv[(i-1) + (j-1)*ldx] with the halo columns at
// i = 1 and i = w+2.
struct Strip {
  const float *arr[6];  // AX, AY, BB, CX, CY, F
  int ld[6];
  int il, inc, seam;
  double *xv;
  int ldx;
  const double *rinv, *rinv1;
  double *dum0;  // (w, nblk-1)
  const int *ie;
  int nblk, w;
  __device__ int col(int c) const {
    c = c < w ? c : 0;
    return (seam && c >= inc) ? c - inc : il - 1 + c;
  }
  __device__ double *xrow(int j) const { return xv + 1 + (long)(j - 1) * ldx; }  // &X(2, j)
};

// IE(k+1) from the LDS copy, as a wave-uniform (scalar) value.
__device__ __forceinline__ int ie_at(const int *ie, int k) { return __builtin_amdgcn_readfirstlane(ie[k]); }

__device__ __forceinline__ int fwd_jlast(const int *ie, int nblk) {
  const int ieb = ie_at(ie, nblk - 1), js = nblk > 1 ? ie_at(ie, nblk - 2) : 1;
  return ieb - 2 >= js ? ieb - 2 : js - 1;
}

// Chunk hand-over.  The marcher's outstanding global loads are influence
// columns for a later closure, so its barrier waits for LDS only; the
// stager's also waits for its DMAs and stores.
__device__ __forceinline__ void bar_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void bar_all() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Lane t's dword of a 64-dword run at dst (wave-uniform) comes from src.
__device__ __forceinline__ void dma(const void *src, uint32_t *dst) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void *)(src),
                                   (__attribute__((address_space(3))) void *)(dst), 4, 0, 0);
}

// The closures' dot products, sum_{m=1..w} e(m) R(m, n), sequential from zero
// (column n for lane n).
//
// Strips up to 32 wide (WMAX = 32) have their rows in the upper half of the
// marching wavefront and the columns in both: lane 32 + n takes the entries
// after the first h = ceil(w / 2) of column n, lane n those, so a column is
// half the loads and a dot product half the multiplies.  The lower half's sum
// goes to the upper half, which adds its terms to it: the additions are the
// sequential ones.  e(m) reaches the lanes by a permutation (lane i of every
// 16-lane row gets entry i of its half's part) and broadcasts within the
// multiply-adds.  A 24-wide closure took 572 clocks with e through LDS and one
// lane a column, and takes about 300.
//
// Wider strips (WMAX = 64) hold a column a lane; e goes through LDS (eb, the
// marcher's own buffer) and comes back as broadcast reads of two entries.
//
// The entries past the column's end that a fixed count loads belong to the
// next column or the allocation's padding and are never used.  WX > 0: the
// strip width is WX, so the loads are exact and the terms unguarded.
template <int WMAX, int WX>
struct Closure {
  static constexpr int NC = WMAX == 32 ? (WX > 0 ? (WX + 1) / 2 : 16) : WMAX;  // entries a lane holds
  int w, lane, h, src;
  uint32_t off;
  double *eb;
  __device__ Closure(int w_, int lane_, int n, double *eb_)
      : w(w_), lane(lane_), h(WX > 0 ? (WX + 1) / 2 : (w_ + 1) / 2),
        src(4 * (32 + (lane_ >> 5) * h + (lane_ & 15))),
        off(8 * (n * w_ + (WMAX == 32 ? (lane_ >> 5) * h : 0))), eb(eb_) {}
  // this lane's part of column n of mat
  __device__ void load(double (&r)[NC], const char *mat) const {
    const double *c = reinterpret_cast<const double *>(mat + off);
#pragma unroll
    for (int m = 0; m < NC; ++m) r[m] = c[m];
  }
  // upper half: the lower half's value; lower half: undefined
  __device__ static double from_lower(double v, double any) {
    const auto a = __builtin_amdgcn_permlane32_swap(__double2loint(any), __double2loint(v), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(__double2hiint(any), __double2hiint(v), false, false);
    return __hiloint2double(b[0], a[0]);
  }
  // p(i) = q(lane i of the row) r(i), i = I..NC-1, four at a time.  The
  // multiply-add onto zero takes the broadcast with it: the zeros are made
  // while q is on its way.  (It turns a product of -0 into +0, which no sum
  // that begins at +0 can tell.)
  template <int I>
  __device__ static void products(double (&p)[NC], double q, const double (&r)[NC]) {
    constexpr int N = NC - I < 4 ? NC - I : 4;
#pragma unroll
    for (int i = 0; i < (N == 4 ? 4 : 1); ++i) p[I + i] = 0.0;
    if constexpr (N == 4)
      asm("s_nop 1\n\t"
          "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_fmac_f64_dpp %1, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_fmac_f64_dpp %2, %4, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_fmac_f64_dpp %3, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf bound_ctrl:1"
          : "+v"(p[I]), "+v"(p[I + 1]), "+v"(p[I + 2]), "+v"(p[I + 3])
          : "v"(q), "v"(r[I]), "v"(r[I + 1]), "v"(r[I + 2]), "v"(r[I + 3]), "n"(I), "n"(I + 1), "n"(I + 2),
            "n"(I + 3));
    else
      asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1"
          : "+v"(p[I]) : "v"(q), "v"(r[I]), "n"(I));
    if constexpr (I + (N == 4 ? 4 : 1) < NC) products<I + (N == 4 ? 4 : 1)>(p, q, r);
  }
  // e to where dot takes it from (the result is dot's first argument)
  __device__ double spread(double e) const {
    if constexpr (WMAX == 32)
      return __hiloint2double(__builtin_amdgcn_ds_bpermute(src, __double2hiint(e)),
                              __builtin_amdgcn_ds_bpermute(src, __double2loint(e)));
    wave_lds_sync();  // the dot product before has read eb
    eb[lane] = e;
    wave_lds_sync();
    return e;
  }
  __device__ double dot(double q, const double (&r)[NC]) const {
    if constexpr (WMAX == 32) {
      double p[NC], s = 0.0;
      products<0>(p, q, r);
#pragma unroll
      for (int i = 0; i < NC; ++i)
        if (WX > 0 || i < h) s = s + p[i];
      s = from_lower(s, q);
#pragma unroll
      for (int i = 0; i < (WX > 0 ? WX / 2 : NC); ++i)
        if (WX > 0 || i < w - h) s = s + p[i];
      return s;
    } else {
      const double2 *e2 = reinterpret_cast<const double2 *>(eb);
      double s = 0.0;
#pragma unroll
      for (int g = 0; g < WMAX / 8; ++g) {
        if (8 * g >= w) break;
        double2 cur[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) cur[i] = e2[4 * g + i];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 8 * g + 2 * i;
          if (m < w) {
            s = s + cur[i].x * r[m];
            if (m + 1 < w) s = s + cur[i].y * r[m + 1];
          }
        }
      }
      return s;
    }
  }
};

// ------------------------------------------------------------ record order
// One record of a pass (an entry of bir_record_table): its kind, block nb,
// row j and the block's IE and JS, all wave-uniform.
struct RecInfo {
  int kind, j, nb, js, ieb;
};

// ------------------------------------------------------------------ stager
template <int WMAX>
struct StagerLane {
  static constexpr int NQ = Stage<WMAX>::NQ;
  // lane t of a quad's DMA d fetches entry t & 3 of column (64 d + t) / 4
  const float *f0[NQ], *f1[NQ];  // AX, AY, BB, CX and CY, F (twice) at row 1
  int ld0, ld1;
  int doff[NQ];  // byte offset of entry t & 1 of a double of the column in its row
  int hoff[NQ];  // the same for the halo: X(1, .) or, at column w, X(w+2, .)
  int poff[Stage<WMAX>::ND];  // hoff for the pair's DMAs
  __device__ void init(const Strip &s, int t) {
    const float *a0 = s.arr[0], *a1 = t & 1 ? s.arr[5] : s.arr[4];
    ld0 = s.ld[0];
    ld1 = t & 1 ? s.ld[5] : s.ld[4];
#pragma unroll
    for (int k = 1; k < 4; ++k)
      if ((t & 3) == k) { a0 = s.arr[k]; ld0 = s.ld[k]; }
#pragma unroll
    for (int d = 0; d < NQ; ++d) {
      const int c = (64 * d + t) / 4, k = min(c, s.w - 1);
      f0[d] = a0 + s.col(c);
      f1[d] = a1 + s.col(c);
      doff[d] = 8 * k + 4 * (t & 1);
      hoff[d] = (k == s.w - 1 ? (s.w + 1) * 8 : 0) + 4 * (t & 1);
    }
#pragma unroll
    for (int e = 0; e < Stage<WMAX>::ND; ++e)
      poff[e] = ((64 * e + t) / 2 >= s.w - 1 ? (s.w + 1) * 8 : 0) + 4 * (t & 1);
  }
};

template <int WMAX>
__device__ __forceinline__ void fill_record(Stage<WMAX> &S, const Strip &s, const StagerLane<WMAX> &L,
                                            int b, int p, const RecInfo &k, int t) {
  using G = Stage<WMAX>;
  uint32_t *rec = S.in[b][p];
  const bool upper = t & 2;  // of the lane's quad: entries 2 and 3
  auto quad0 = [&](int j) {
#pragma unroll
    for (int d = 0; d < G::NQ; ++d) dma(L.f0[d] + (long)(j - 1) * L.ld0, rec + 64 * d);
  };
  // entries 0 and 1 from the coefficient rows j, 2 and 3 from a row of doubles
  auto quad1 = [&](int j, const double *row, const int (&off)[G::NQ]) {
#pragma unroll
    for (int d = 0; d < G::NQ; ++d) {
      const char *f = (const char *)(L.f1[d] + (long)(j - 1) * L.ld1);
      dma(upper ? (const char *)row + off[d] : f, rec + 4 * WMAX + 64 * d);
    }
  };
  auto rows2 = [&](const double *r0, const double *r1) {  // quad 0: two rows of doubles
    const char *r = (const char *)(upper ? r1 : r0);
#pragma unroll
    for (int d = 0; d < G::NQ; ++d) dma(r + L.doff[d], rec + 64 * d);
  };
  auto halo = [&](int j) {
#pragma unroll
    for (int e = 0; e < G::ND; ++e)
      dma((const char *)(s.xv + (long)(j - 1) * s.ldx) + L.poff[e], rec + 8 * WMAX + 64 * e);
  };
  // The record's influence matrix into this XCD's L2, a line a lane: the
  // marcher loads its columns a block ahead of the closure, about the time of
  // an L2 hit and half that of the memory behind it.
  auto touch = [&](const double *mat) {
    const int n = s.w * s.w * 8;
#pragma unroll
    for (int q = 0; q < WMAX * WMAX * 8 / (64 * 128); ++q) {  // 8 KiB an instruction
      const int o = 128 * (64 * q + t);
      if (o < n) dma((const char *)mat + o, S.touched);
    }
  };
  const double *xr = (k.nb != s.nblk) ? s.dum0 + (long)(k.nb - 1) * s.w : s.xrow(k.ieb);
  switch (k.kind) {
    case BIR_HEAD:
      rows2(s.xrow(1), s.xrow(2));
      break;
    case BIR_ROW:
      quad0(k.j);
      quad1(k.j, s.xv + (long)k.j * s.ldx, L.hoff);  // X(., j+1)
      break;
    case BIR_CLOS:
      quad0(k.j);
      quad1(k.j, s.xrow(k.ieb + 1), L.doff);
      halo(k.j + 1);
      touch(s.rinv1 + (long)(k.nb - 1) * s.w * s.w);
      break;
    case BIR_A:
      quad0(k.ieb - 1);
      quad1(k.ieb - 1, xr, L.doff);
      halo(k.ieb);
      touch(s.rinv + (long)(k.nb - 1) * s.w * s.w);
      break;
    case BIR_B:
      // with a one-row block X(., JS+1) is row IE, read after its restore
      rows2(s.xrow(k.ieb - 1), k.js + 1 == k.ieb ? xr : s.xrow(k.js + 1));
      quad1(max(k.js - 1, 1), k.nb == s.nblk ? s.xrow(k.ieb + 1) : xr, L.doff);
      if (k.nb != 1) touch(s.rinv1 + (long)(k.nb - 2) * s.w * s.w);
      break;
    default:  // BIR_BROW: the last row reads row IE after its restore
      quad0(k.j);
      quad1(k.j, k.j + 2 == k.ieb ? xr : s.xrow(k.j + 2), L.doff);
      break;
  }
}

// The record's results to memory.  The destination rows are wave-uniform and
// chosen first; only the stores themselves are limited to the strip's lanes.
template <int WMAX>
__device__ __forceinline__ void drain_record(Stage<WMAX> &S, const Strip &s, int b, int p,
                                             const RecInfo &k, int t, double o0) {
  double *d0 = nullptr, *d1 = nullptr, *dr = nullptr;
  if (k.kind == BIR_ROW) {  // row IE(nb) of a closing block waits for its correction
    if (!(k.nb < s.nblk && k.j == k.ieb - 2)) d0 = s.xrow(k.j + 2);
  } else if (k.kind == BIR_CLOS) {
    d0 = s.xrow(k.ieb);
    d1 = s.dum0 + (long)(k.nb - 1) * s.w;
  } else if (k.kind == BIR_B) {
    // restore row IE from DUM0 (still in the record); a block with march
    // rows overwrites it with its last row, so only a one-row block keeps it
    if (k.nb != s.nblk && k.ieb - 2 < k.js) dr = s.xrow(k.ieb);
    d0 = s.xrow(k.js + 1);
  } else if (k.kind == BIR_BROW) {
    d0 = s.xrow(k.j + 2);
  }
  const bool act = t < s.w;
  if (dr && act) dr[t] = *reinterpret_cast<const double *>(&S.in[b][p][4 * WMAX + 4 * t + 2]);
  if (d0 && act) d0[t] = o0;
  if (d1 && act) d1[t] = *reinterpret_cast<const double *>(&S.in[b][p][2 * t]);
}

// One pass for stager `sid`: it fills and drains the records p of each chunk
// with p % NSTG == sid.  The record-table entries of each chunk come into an
// LDS ring by DMA two chunks ahead: stager 0 issues them, except the first two
// chunks' entries, which every stager loads for itself.  Records of one pass read only rows
// that no record of the same pass writes, and write distinct rows, so the
// stagers need no ordering among themselves inside a pass; the barrier after
// the last drain makes every result visible to the next pass's DMAs.
template <int WMAX>
__device__ void stage_pass(Stage<WMAX> &S, const Strip &s, const StagerLane<WMAX> &L, int t, int sid,
                           bool fwd, const int *recs) {
  constexpr int R = Stage<WMAX>::R;
  const int T = fwd ? 1 + fwd_jlast(s.ie, s.nblk) : s.nblk + ie_at(s.ie, s.nblk - 1) - 1;
  const int C = (T + R - 1) / R;
  auto load_desc = [&](int c) {
#pragma unroll
    for (int k = 0; k < (R * 4 + 63) / 64; ++k)
      if (64 * k + t < R * 4)
        dma(recs + (long)c * R * 4 + 64 * k + t, reinterpret_cast<uint32_t *>(&S.desc[c & 3][0][0]) + 64 * k);
  };
  // This stager's entries of chunk c, one per lane (lane i: record sid +
  // i*NSTG), read at once; the i-th is then taken with lane reads.
  auto descs = [&](int c, int n) {
    const int p = sid + NSTG * t;
    int4 d = make_int4(0, 0, 0, 0);
    if (p < n) d = *reinterpret_cast<const int4 *>(S.desc[c & 3][p]);
    return d;
  };
  auto cur_at = [&](const int4 &d, int i) {
    RecInfo k;
    const int kn = __builtin_amdgcn_readlane(d.x, i);
    k.kind = kn & 255;
    k.nb = kn >> 8;
    k.j = __builtin_amdgcn_readlane(d.y, i);
    k.ieb = __builtin_amdgcn_readlane(d.z, i);
    k.js = __builtin_amdgcn_readlane(d.w, i);
    return k;
  };
  auto fill = [&](int c) {
    const int n = min(R, T - c * R);
    const int4 d = descs(c, n);
    for (int i = 0, p = sid; p < n; ++i, p += NSTG) fill_record<WMAX>(S, s, L, c % 3, p, cur_at(d, i), t);
  };
  // Each result is read from LDS a record ahead of its store.
  auto drain = [&](int c) {
    const int n = min(R, T - c * R);
    const int4 d = descs(c, n);
    const int tl = t & (WMAX - 1);
    auto result = [&](int p) { return *reinterpret_cast<const double *>(&S.in[c % 3][p][8 * WMAX + 2 * tl]); };
    double on = sid < n ? result(sid) : 0.0;
    for (int i = 0, p = sid; p < n; ++i, p += NSTG) {
      const double o0 = on;
      if (p + NSTG < n) on = result(p + NSTG);
      drain_record<WMAX>(S, s, c % 3, p, cur_at(d, i), t, o0);
    }
  };
  load_desc(0);
  if (C > 1) load_desc(1);
  wait_vm();
  fill(0);
  bar_all();
  for (int c = 0; c < C; ++c) {
    if (sid == 0 && c + 2 < C) load_desc(c + 2);
    if (c + 1 < C) fill(c + 1);
    if (c >= 1) drain(c - 1);
    bar_all();
  }
  drain(C - 1);
  bar_all();  // pass end
}

// ----------------------------------------------------------------- marcher
struct Rec {
  uint4 q0, q1;
  uint2 pr;
  __device__ static double f(uint32_t v) { return (double)__uint_as_float(v); }
  __device__ static double d(uint32_t lo, uint32_t hi) { return __hiloint2double((int)hi, (int)lo); }
  __device__ double a() const { return f(q0.x); }
  __device__ double b() const { return f(q0.y); }
  __device__ double c() const { return f(q0.z); }
  __device__ double dd() const { return f(q0.w); }
  __device__ double e() const { return f(q1.x); }
  __device__ double ff() const { return f(q1.y); }
  __device__ double row0() const { return d(q0.x, q0.y); }
  __device__ double row1() const { return d(q0.z, q0.w); }
  __device__ double y() const { return d(q1.z, q1.w); }
  __device__ double halo() const { return d(pr.x, pr.y); }
};

// The marcher's walk through the records: two lane addresses advance by one
// record per step and wrap with the buffers at chunk ends.  The marching
// wavefront issues an instruction in five clocks, a branch in 12 or, taken, 24,
// so the walk is kept to few: wide reads at constant offsets from an address,
// results written into the record they replace, one way through a record.
template <int WMAX>
struct MarchIO {
  using G = Stage<WMAX>;
  static constexpr int R = G::R;
  static constexpr int RB = G::REC * 4;  // bytes per record
  static constexpr int PAIR = 32 * WMAX;  // the pair's offset in a record
  char *q, *r;  // the current record's quads and pair, at this lane
  int left = R, buf = 0;
  __device__ MarchIO(G &s, int wlane)
      : q(reinterpret_cast<char *>(&s.in[0][0][4 * (wlane & (WMAX - 1))])),
        r(reinterpret_cast<char *>(&s.in[0][0][8 * WMAX + 2 * (WMAX == 32 ? wlane ^ 32 : wlane)])) {}
  __device__ void read(Rec &c, int o) {
    c.q0 = *reinterpret_cast<const uint4 *>(q + o);
    c.q1 = *reinterpret_cast<const uint4 *>(q + o + 16 * WMAX);
    c.pr = *reinterpret_cast<const uint2 *>(r + o);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ void start(Rec &c) {
    bar_lds();
    // The columns requested before the barrier have landed by now.  Said so
    // that the compiler knows: a load it believes in flight makes every later
    // write to the registers it used wait for all loads, in the loops too.
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    read(c, 0);
  }
  // The next record (past the third buffer's end what lies beyond it: a
  // discarded prefetch), once v, all that is wanted of the current one, is
  // made: c's registers are free, and the division or dot product that
  // follows covers the reads.  The barriers keep the reads here: left to
  // itself the compiler moves them down to their use, behind the branches.
  __device__ static void made(double &v) { asm volatile("" : "+v"(v) : : "memory"); }
  __device__ void fetch(Rec &c, double &v) {
    made(v);
    read(c, RB);
  }
  __device__ void put(double v) { *reinterpret_cast<double *>(r) = v; }
  __device__ void put2(double v) { *reinterpret_cast<double *>(r - PAIR) = v; }
  // After the record: at the chunk's end its barrier, then the new chunk's
  // first record into c.
  __device__ void next(Rec &c) {
    q += RB;
    r += RB;
    if (__builtin_expect(--left == 0, 0)) {
      bar_lds();
      left = R;
      if (++buf == G::NIN) {
        buf = 0;
        q -= G::NIN * R * RB;
        r -= G::NIN * R * RB;
      }
      read(c, 0);
    }
  }
  // The last chunk's barrier, then the pass-end barrier that waits for the
  // stagers' last results to reach memory.
  __device__ void finish() {
    if (left != R) bar_lds();
    bar_lds();
  }
};

// REPBIR on one strip (MAIN/template/GLOBAL/src/sevp.f90:218-328), consuming
// the forward and backward record sequences.  WX > 0: the strip width is WX.
// With WMAX = 32 the strip's rows are in the upper half of the wavefront
// (lane = strip column - 1 + 32); the lower half computes along on values
// that nothing reads but its part of the closures' dot products, and stores
// its results beside.  A wave shift carries a lane from the lower half only
// into the strip's first column, which takes its halo instead.
template <int WMAX, int WX>
__device__ void march_strip(Stage<WMAX> &S, const Strip &s, int wlane) {
  const int w = s.w, nblk = s.nblk;
  const int lane = wlane & (WMAX - 1);
  const int ww = 8 * w * w;  // bytes per influence matrix
  const Closure<WMAX, WX> cl(w, wlane, lane < w ? lane : 0, S.e);
  double rc[Closure<WMAX, WX>::NC], rc2[Closure<WMAX, WX>::NC];
  Rec c, cb;  // the current record; a backward block's record B
  auto shifts = [&](double x, double h, double &xw, double &xe) {
    xw = wave_shr1_zero(x);
    if (lane == 0) xw = h;
    xe = wave_shl1_zero(x);
    if (lane == w - 1) xe = h;
  };

  // ---------------- forward ----------------
  // Each column array has one load in its loop, a block ahead of the closure
  // that uses it, and the loop one exit, at its end: so the columns stay in
  // the registers they are loaded to and nothing waits for them before.
  const char *m1 = (const char *)s.rinv1, *const mb = (const char *)s.rinv + (long)(nblk - 1) * ww;
  cl.load(rc, nblk > 1 ? m1 : mb);
  double xs, xc;
  auto frows = [&](MarchIO<WMAX> &io, int n) {
    for (; n > 0; --n) {
      double xw, xe;
      shifts(xc, c.y(), xw, xe);  // lane 0: X(1, J+1); lane w-1: X(w+2, J+1)
      const double at = c.e();
      double num = c.ff() - c.a() * xw - c.b() * xs - c.c() * xc - c.dd() * xe;
      io.fetch(c, num);
      xs = xc;
      xc = num / at;
      io.put(xc);
      io.next(c);
    }
  };
  {
    MarchIO<WMAX> io(S, wlane);
    io.start(c);
    const int jlast = fwd_jlast(s.ie, nblk);  // the stagers write s.ie before the first barrier
    xs = c.row0();
    xc = c.row1();
    io.fetch(c, xc);
    io.next(c);
    int js = 1, iev = s.ie[0];
    for (int nb = 1; nb < nblk; ++nb) {
      const int ieb = __builtin_amdgcn_readfirstlane(iev);
      iev = s.ie[nb];  // a block ahead
      frows(io, ieb - 1 - js);
      // residual of the block at row IE-1, correction of row IE
      double xw, xe;
      shifts(xc, c.halo(), xw, xe);
      const double xnn = c.y();
      double res = c.ff() - c.a() * xw - c.b() * xs - c.c() * xc - c.dd() * xe - c.e() * xnn;
      io.made(res);
      const double q = cl.spread(res);
      io.read(c, MarchIO<WMAX>::RB);
      xs = xc - cl.dot(q, rc);
      io.put(xs);
      io.put2(xc);  // DUM0
      xc = xnn;
      io.next(c);
      js = ieb;
      // after the last closure: the backward pass's first block
      m1 += ww;
      cl.load(rc, nb + 1 < nblk ? m1 : mb);
    }
    frows(io, jlast + 1 - js);
    io.finish();
  }
  // one block: no RINV1, its columns unused
  const char *r2 = nblk > 1 ? (const char *)s.rinv1 + (long)(nblk - 2) * ww : mb, *r1 = mb;
  cl.load(rc2, r2);

  // ---------------- backward ----------------
  MarchIO<WMAX> io(S, wlane);
  io.start(c);
  double xnn = 0.0;  // X(., IE+1): the block above's corrected row JS+1
  int iebk = ie_at(s.ie, nblk - 1), jsv = s.ie[max(nblk - 2, 0)];
  for (int nb = nblk; nb >= 1; --nb) {
    const int jsb = nb > 1 ? __builtin_amdgcn_readfirstlane(jsv) : 1;
    jsv = s.ie[max(nb - 3, 0)];  // the next block's JS, a block ahead
    io.read(cb, MarchIO<WMAX>::RB);
    const double xrow = c.y(), an = c.e();
    double xw, xe;
    shifts(xrow, c.halo(), xw, xe);
    double r0 = c.ff() - c.a() * xw;
    const double ab = c.b(), tc = c.c() * xrow, te = c.dd() * xe;
    io.next(cb);
    if (nb == nblk) xnn = cb.y();
    double res = r0 - ab * cb.row0() - tc - te - an * xnn;
    const double xf = cb.row1(), cy = cb.e();
    io.made(res);
    const double q = cl.spread(res);
    io.read(c, MarchIO<WMAX>::RB);
    double hc = cl.dot(q, rc), hs = 0.0;
    xnn = xf + hc;
    io.put(xnn);
    if (__builtin_expect(nb != 1, 1)) hs = cl.dot(cl.spread(hc * cy), rc2);
    io.next(c);
    // the next block's matrices, a block ahead (the first's again at the end)
    if (nb > 1) r1 -= ww;
    if (nb > 2) r2 -= ww;
    cl.load(rc, r1);
    cl.load(rc2, r2);
    for (int n = iebk - 1 - jsb; n > 0; --n) {
      double hw = wave_shr1_zero(hc), he = wave_shl1_zero(hc);
      if (WMAX == 32 && lane == 0) hw = 0.0;  // not the lower half's
      if (lane == w - 1) he = 0.0;
      const double at = c.e(), xo = c.y();
      double num = -(c.a() * hw) - c.b() * hs - c.c() * hc - c.dd() * he;
      io.fetch(c, num);
      hs = hc;
      hc = num / at;
      io.put(xo + hc);
      io.next(c);
    }
    iebk = jsb;
  }
  io.finish();
}

// ----------------------------------------------------------------- kernels
// The block rows IE live in LDS for the whole launch: every stager copies
// them (the same values) before its first chunk, so neither the marcher, which
// reads them only after the first chunk barrier, nor the stagers wait on
// global memory for them.
__device__ inline void load_ie(int *dst, const int *src, int nblk, int t) {
  for (int b = t; b < nblk; b += SEVP_WAVE) dst[b] = src[b];
  wait_vm();
}

__device__ inline Strip bir_strip(const BirArgs &p, const int *ie, int r, int n) {
  Strip s;
  const int w = p.ibir, inc = p.ibir / 2;
  const int i0 = p.i2 + 2;
  const int il = (n - 1) * inc + 1;
  s.arr[0] = p.al; s.arr[1] = p.ab; s.arr[2] = p.ac; s.arr[3] = p.ar; s.arr[4] = p.at;
  s.arr[5] = p.s + (long)r * p.s_stride;
  for (int k = 0; k < 6; ++k) s.ld[k] = p.i2;
  s.il = il;
  s.inc = inc;
  s.seam = n == p.nbir;
  if (!s.seam) {
    s.xv = p.x + (long)r * p.x_stride + f2(i0, il, 1);
    s.ldx = i0;
  } else {
    s.xv = p.xx + (long)r * p.xx_stride;
    s.ldx = w + 2;
  }
  const long ibr2 = (long)w * w;
  s.rinv = p.rinv + (long)(n - 1) * ibr2 * p.nb0;
  s.rinv1 = p.rinv1 + (long)(n - 1) * ibr2 * (p.nb0 - 1);
  s.dum0 = p.dum0 + (long)r * p.dum0_stride;
  s.ie = ie;
  s.nblk = p.nb0;
  s.w = w;
  return s;
}

// Whole FS_SOLVER BIR loop (MAIN/template/GLOBAL/src/fs_GLOBAL.f90:1902-1966)
// for one RHS per workgroup.  The seam strip's halo gather and write-back
// (and the periodic halo refresh) are done by every stager in full: the
// stagers write identical values, and each reads only what it has itself
// written before its next pass's DMAs.
template <int WMAX, int WX>
__global__ __launch_bounds__(BIR_THREADS) void bir_sweeps_kernel(BirArgs p) {
  __shared__ Stage<WMAX> S;
  __shared__ int ie[BIR_MAX_BLOCKS];
  const int r = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = threadIdx.x & 63;
  if (wave == 0) {
    for (int it = 0; it < p.nsweep; ++it)
      for (int n = 1; n <= p.nbir; ++n) march_strip<WMAX, WX>(S, bir_strip(p, ie, r, n), t);
    return;
  }
  const int sid = wave - 1;
  load_ie(ie, p.ie, p.nb0, t);
  const int w = p.ibir, inc = p.ibir / 2;
  const int i0 = p.i2 + 2, m0 = w + 2;
  const int j1 = p.j2 + 1;
  double *x = p.x + (long)r * p.x_stride;
  double *xx = p.xx + (long)r * p.xx_stride;
  for (int it = 0; it < p.nsweep; ++it) {
    for (int n = 1; n <= p.nbir; ++n) {
      const Strip s = bir_strip(p, ie, r, n);
      const int il = s.il;
      if (s.seam) {
        // seam strip: halo columns of XX for rows 1..J2 as the reference does
        // (row J1 keeps its old value), or 1..J1 with seam_fix
        const int jg = p.seam_fix ? j1 : p.j2;
        for (int j = 1 + t; j <= jg; j += SEVP_WAVE) {
          xx[f2(m0, 1, j)] = x[f2(i0, il, j)];
          xx[f2(m0, w + 2, j)] = x[f2(i0, inc + 2, j)];
        }
        wait_vm();
      }
      StagerLane<WMAX> L;
      L.init(s, t);
      stage_pass<WMAX>(S, s, L, t, sid, true, p.recs);
      stage_pass<WMAX>(S, s, L, t, sid, false, p.recs + 4L * p.fwd_records);
      if (s.seam) {
        for (long q = t; q < (long)w * (j1 - 1); q += SEVP_WAVE) {
          const int i = (int)(q % w) + 1, j = (int)(q / w) + 2;
          const double v = xx[f2(m0, i + 1, j)];
          if (i <= inc) x[f2(i0, il + i, j)] = v;
          else x[f2(i0, i - inc + 1, j)] = v;
        }
        wait_vm();
        if (p.periodic) {
          for (int j = 2 + t; j <= j1; j += SEVP_WAVE) {
            x[f2(i0, 1, j)] = x[f2(i0, i0 - 1, j)];
            x[f2(i0, i0, j)] = x[f2(i0, 2, j)];
          }
          wait_vm();
        }
      }
    }
  }
}

// One REPBIR call with the reference's argument conventions, batched over
// independent right-hand sides (F and X strided by f_stride / x_stride).
template <int WMAX, int WX>
__global__ __launch_bounds__(BIR_THREADS) void repbir_kernel(RepbirArgs p) {
  __shared__ Stage<WMAX> S;
  __shared__ int ie[BIR_MAX_BLOCKS];
  const int r = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = threadIdx.x & 63;
  Strip s;
  s.arr[0] = p.ax; s.arr[1] = p.ay; s.arr[2] = p.bb; s.arr[3] = p.cx; s.arr[4] = p.cy;
  s.arr[5] = p.f + (long)r * p.f_stride;
  for (int k = 0; k < 5; ++k) s.ld[k] = p.i2;
  s.ld[5] = p.m2;
  s.il = 1;
  s.inc = 0;
  s.seam = 0;
  s.xv = p.x + (long)r * p.x_stride;
  s.ldx = p.i0;
  s.rinv = p.rinv;
  s.rinv1 = p.rinv1;
  s.dum0 = p.dum0 + (long)r * p.dum0_stride;
  s.ie = ie;
  s.nblk = p.nblk;
  s.w = p.m2;
  if (wave == 0) {
    march_strip<WMAX, WX>(S, s, t);
    return;
  }
  load_ie(ie, p.ie, p.nblk, t);
  StagerLane<WMAX> L;
  L.init(s, t);
  stage_pass<WMAX>(S, s, L, t, wave - 1, true, p.recs);
  stage_pass<WMAX>(S, s, L, t, wave - 1, false, p.recs + 4L * p.fwd_records);
}

// Strips of width 24 and 30 (the 0.5, 0.25 and 0.1 degree configurations)
// run kernels specialised for their width.
hipError_t launch_bir_sweeps(const BirArgs &a, int nrhs, hipStream_t st) {
  const dim3 g(nrhs), b(BIR_THREADS);
  if (a.ibir == 24) hipLaunchKernelGGL((bir_sweeps_kernel<32, 24>), g, b, 0, st, a);
  else if (a.ibir == 30) hipLaunchKernelGGL((bir_sweeps_kernel<32, 30>), g, b, 0, st, a);
  else if (a.ibir <= 32) hipLaunchKernelGGL((bir_sweeps_kernel<32, 0>), g, b, 0, st, a);
  else hipLaunchKernelGGL((bir_sweeps_kernel<64, 0>), g, b, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_repbir(const RepbirArgs &a, int nrhs, hipStream_t st) {
  const dim3 g(nrhs), b(BIR_THREADS);
  if (a.m2 == 24) hipLaunchKernelGGL((repbir_kernel<32, 24>), g, b, 0, st, a);
  else if (a.m2 == 30) hipLaunchKernelGGL((repbir_kernel<32, 30>), g, b, 0, st, a);
  else if (a.m2 <= 32) hipLaunchKernelGGL((repbir_kernel<32, 0>), g, b, 0, st, a);
  else hipLaunchKernelGGL((repbir_kernel<64, 0>), g, b, 0, st, a);
  return hipGetLastError();
}

}  // namespace sevp

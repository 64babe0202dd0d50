// Where the fused pass's workgroups and matrix columns are: plain C++ with no
// HIP dependency, so that host tests can build it alone.
#pragma once

#ifdef __HIPCC__
#define SEVP_HD __host__ __device__ __forceinline__
#else
#define SEVP_HD inline
#endif

namespace sevp {

// XCD-aware placement: workgroup id -> (column tile, 16-row block).  The
// dispatcher deals workgroups to the 8 XCDs in turn; the row blocks of one
// column tile get ids that land on the same XCD, tile % 8, one after another.
// Each part of a launch (homogeneous march, products, next matrices) begins at
// a multiple of 8, so this holds in every part of every launch.
SEVP_HD bool tile_of(int wg, int ntiles, int nmb, int &tile, int &mb) {
  const int xcd = wg & 7, slot = wg >> 3;
  tile = (slot / nmb) * 8 + xcd;
  mb = slot % nmb;
  return tile < ntiles;
}
SEVP_HD long placed_workgroups(int ntiles, int nmb) { return 8L * nmb * ((ntiles + 7) / 8); }
// Workgroups of `waves` wavefronts' work, w each, to the next multiple of 8.
SEVP_HD int march_workgroups(long waves, int w) { return (int)((waves + 8L * w - 1) / (8L * w) * 8); }

// Forward tiles are of 16 columns, of which 16 - 2 steps are written.
SEVP_HD int fused_tiles_fwd(int i2, int steps) {
  const int tout = 16 - 2 * steps;
  return tout > 0 ? (i2 + tout - 1) / tout : 0;
}
// Tile column i (0..15) of a forward tile: the interior column (1-based,
// before wrapping), and the one whose matrix column is read for it.
SEVP_HD int fused_fwd_column(int tile, int steps, int i) { return tile * (16 - 2 * steps) - steps + 1 + i; }
SEVP_HD int fused_fwd_matrix_column(int c, int i2, int periodic) {
  if (periodic) return ((c - 1) % i2 + i2) % i2 + 1;
  return c < 1 ? 1 : (c > i2 ? i2 : c);
}

// Workgroup wg of the part of a launch that brings the next launch's matrices
// near: the column tile of the next launch whose columns it reads.  Its XCD is
// the tile's; a forward launch's tiles are those of the next block's steps.
SEVP_HD bool warm_tile(int wg, int ntiles_next, int &tile) {
  int mb;
  return tile_of(wg, ntiles_next, 1, tile, mb);
}

}  // namespace sevp

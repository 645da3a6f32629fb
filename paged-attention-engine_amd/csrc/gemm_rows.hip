// Products of up to 16 rows: which kernel of gemm_rows_kernel.h takes one, and those that take 16 weight rows a workgroup.
#include "gemm_rows_kernel.h"

// Whether workgroups take eight weight rows instead of 16: by the rows of W and A that the busiest of the 256 compute units has to take in, which bounds
// these products.  Eights count for less, 0.85: more of them are under way beside each other.  Us at 4 / 8 / 16 rows, eights and sixteens: 128
// tiles of 1,536 of k 5.1 / 5.3 / 5.9 and 5.5 / 5.8 / 6.5, 160 of 2,048 6.5 / 7.0 / 7.9 and 6.3 / 6.6 / 7.4, 288 of 3,584 10.4 / 11.2 / 13.8 and 11.2 / 11.9 / 13.7,
// 448 of 5,120 17.5 / 20.1 / 24.5 and 16.9 / 18.3 / 20.6, 608 of 896 6.5 / 6.9 / 8.0 and 6.9 / 7.1 / 7.9, 1,120 of 1,536 12.3 / 13.8 / 17.6 and 12.6 / 13.2 /
// 15.0, 1,376 of 2,048 18.1 / 20.4 / 25.1 and 19.6 / 20.4 / 23.6.
static bool takes_halves(int tiles, int groups) {
  const int64_t of_a = 4 * groups, whole = (tiles + 255) / 256 * (16 + of_a), halves = (2 * (int64_t)tiles + 255) / 256 * (8 + of_a);
  return 17 * halves <= 20 * whole;
}

int launch_rows(const RowsProduct& p, hipStream_t stream) {
  const int tiles = (p.N + 15) / 16;
  const int groups = p.M <= 4 ? 1 : p.M <= 8 ? 2 : p.M <= 12 ? 3 : 4;
  int k_per_range = (p.K + p.splits - 1) / p.splits;
  k_per_range = (k_per_range + 127) / 128 * 128;
  // a share of the sums of squares may cover 16 weight rows: then a workgroup has to
  const bool whole_tiles = p.epilogue == EPI_RESIDUAL && p.norm.next_stat_tiles < 2 * tiles;
  if (p.epilogue == EPI_RESIDUAL && (p.splits == 2 || (p.splits == 4 && !whole_tiles))) {  // side by side in one workgroup
    // (sixteen wavefronts of 16 weight rows have no registers for more than eight rows of A: four ranges of whole tiles go by ticket)
    if (!whole_tiles) {
      launch_rows_halves(p, p.splits, k_per_range, dim3(2 * tiles), stream);
    } else {
      switch (groups) {
        case 1: launch_rows_of<4, 1, 8, 1>(p, k_per_range, dim3(tiles), stream); break;
        case 2: launch_rows_of<4, 2, 8, 1>(p, k_per_range, dim3(tiles), stream); break;
        case 3: launch_rows_of<4, 3, 8, 1>(p, k_per_range, dim3(tiles), stream); break;
        default: launch_rows_of<4, 4, 8, 1>(p, k_per_range, dim3(tiles), stream); break;
      }
    }
    return pae_check_launch("gemm_rows (ranges side by side)");
  }
  if (p.splits == 1 && p.M <= 16 && !whole_tiles && takes_halves(tiles, groups)) {
    launch_rows_halves(p, 1, k_per_range, dim3(2 * tiles), stream);
  } else {
    // more than 16 rows are shared out by 16, or by 8 where workgroups are few even so (1,536 x 1,536 at 17 rows 4.65 -> 4.46 us, 896 x 896 3.63 -> 3.24)
    if (p.M > 16 && (int64_t)tiles * p.splits * ((p.M + 7) / 8) <= 320) {
      launch_rows_of<4, 2, 4, 1>(p, k_per_range, dim3(tiles, p.splits, (p.M + 7) / 8), stream);
      return pae_check_launch("gemm_rows (rows of A by eight)");
    }
    const dim3 grid(tiles, p.splits, (p.M + 15) / 16);
    switch (groups) {
      case 1: launch_rows_of<4, 1, 4, 2>(p, k_per_range, grid, stream); break;
      case 2: launch_rows_of<4, 2, 4, 1>(p, k_per_range, grid, stream); break;
      case 3: launch_rows_of<4, 3, 4, 1>(p, k_per_range, grid, stream); break;
      default: launch_rows_of<4, 4, 4, 1>(p, k_per_range, grid, stream); break;
    }
  }
  return pae_check_launch("gemm_rows");
}

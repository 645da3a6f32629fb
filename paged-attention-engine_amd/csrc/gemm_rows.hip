// Products of up to 16 rows: which kernel of gemm_rows_kernel.h takes one, and those that take 16 weight rows a workgroup.
#include "gemm_rows_kernel.h"

// Whether workgroups take eight weight rows instead of 16: by the rows of W and A that the busiest of the 256 compute units has to take in, which bounds
// these products.  Eights count for less, 0.85, as more of them are under way beside each other, 0.75 where all of k is asked for at once in four steps and units have two or more;
// and with one workgroup a unit and batches of steps (k above 2,048) eights always have more under way.  Measured with the gate at five k from 896 to 3,584
// by 16 numbers of tiles from 96 to 2,368 and 1 to 16 rows, the rule is 0.2 % behind the faster of the two on average and 8.5 % at worst.  Us at 4 / 8 / 16
// rows, eights and sixteens: 96 tiles of 1,536 of k 3.9 / 3.9 / 4.1 and 4.0 / 4.1 / 4.7, 192 of 1,536 5.2 / 5.4 / 6.1 and 5.0 / 5.1 / 5.6, 192 of 3,584 7.5 / 7.9 /
// 9.9 and 7.5 / 7.8 / 11.5, 320 of 3,584 10.1 / 10.6 / 12.6 and 10.9 / 11.1 / 13.9, 512 of 2,048 8.9 / 9.1 / 11.0 and 9.5 / 9.6 / 10.4, 1,120 of 1,536 12.3 /
// 13.1 / 16.4 and 12.7 / 12.6 / 14.1, 2,368 of 3,584 48.4 / 51.5 / 65.5 and 49.5 / 50.0 / 57.8.
static bool takes_halves(int tiles, int groups, int K) {
  if (tiles <= 256 && K > 2048) return true;
  const int64_t of_a = 4 * groups, whole = (tiles + 255) / 256 * (16 + of_a), halves = (2 * (int64_t)tiles + 255) / 256 * (8 + of_a);
  return (K > 1536 && K <= 2048 && tiles > 192 ? 15 : 17) * halves <= 20 * whole;
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
  if (p.splits == 1 && p.M <= 16 && !whole_tiles && takes_halves(tiles, groups, p.K)) {
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

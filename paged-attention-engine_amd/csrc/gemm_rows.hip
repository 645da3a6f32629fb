// Products of up to 16 rows: which kernel of gemm_rows_kernel.h takes one, and those that take 16 weight rows a workgroup.
#include "gemm_rows_kernel.h"

int launch_rows(const RowsProduct& p, hipStream_t stream) {
  const int tiles = (p.N + 15) / 16;
  const int groups = p.M <= 4 ? 1 : p.M <= 8 ? 2 : p.M <= 12 ? 3 : 4;
  int k_per_range = (p.K + p.splits - 1) / p.splits;
  k_per_range = (k_per_range + 127) / 128 * 128;
  // a share of the sums of squares may cover 16 weight rows: then a workgroup has to
  const bool whole_tiles = p.epilogue == EPI_RESIDUAL && p.norm.next_stat_tiles < 2 * tiles;
  if ((p.splits == 2 || p.splits == 4) && p.epilogue == EPI_RESIDUAL) {  // side by side in one workgroup
    // (one round of 16-row workgroups over the chip: 7B down at 8 / 16 rows 25.2 / 31.7 us, in halves 30.0 / 38.0; else halves, 3B down 14.1 / 18.4
    // against 11.9 / 14.1, 14B O 14.2 / 18.6 against 13.4 / 16.3)
    const bool halves = !whole_tiles && !(tiles > 200 && tiles <= 256 && groups > 1);
    if (halves) {
      launch_rows_halves(p, p.splits, k_per_range, dim3(2 * tiles), stream);
    } else if (p.splits == 4) {  // (sixteen wavefronts have no registers for more than eight rows of A)
      if (groups == 1) launch_rows_of<4, 1, 16, 1>(p, k_per_range, dim3(tiles), stream);
      else launch_rows_of<4, 2, 16, 1>(p, k_per_range, dim3(tiles, 1, (p.M + 7) / 8), stream);
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
  // Eight weight rows a workgroup where workgroups are few, and, up to four rows of A, always (1.5B gate/up 12.1 -> 11.7 us, QKV 4.2 ->
  // 3.8); with more rows their second share of A's fragments costs more (gate/up at 8 / 16 rows 13.4 / 16.3 -> 14.4 / 21.1; 0.5B gate/up, 608
  // tiles, at 9 rows 8.6 -> 7.9, at 16 9.3 -> 8.9; 1.5B up, 560 tiles, 8.9 -> 8.5 and 9.7 -> 11.0).
  const bool halves = p.splits == 1 && p.M <= 16 && !whole_tiles && (groups == 1 || tiles <= (groups == 4 ? 400 : 640));
  if (halves) {
    launch_rows_halves(p, 1, k_per_range, dim3(2 * tiles), stream);
  } else {
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

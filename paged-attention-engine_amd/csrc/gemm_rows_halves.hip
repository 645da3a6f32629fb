// The kernels of gemm_rows.hip that take eight weight rows a workgroup.
#include "gemm_rows_kernel.h"

void launch_rows_halves(const RowsProduct& p, int side_by_side, int k_per_range, dim3 grid, hipStream_t stream) {
  const int groups = p.M <= 4 ? 1 : p.M <= 8 ? 2 : p.M <= 12 ? 3 : 4;
#define ROWS_HALVES(NW, U1, U2, U3)                                                   \
  switch (groups) {                                                               \
    case 1: launch_rows_of<2, 1, NW, U1>(p, k_per_range, grid, stream); break;    \
    case 2: launch_rows_of<2, 2, NW, U2>(p, k_per_range, grid, stream); break;    \
    case 3: launch_rows_of<2, 3, NW, U3>(p, k_per_range, grid, stream); break;     \
    default: launch_rows_of<2, 4, NW, U3>(p, k_per_range, grid, stream); break;    \
  }
  if (side_by_side == 4) {
    ROWS_HALVES(16, 1, 1, 1)
  } else if (side_by_side == 2) {
    ROWS_HALVES(8, 2, 2, 1)
  } else if (grid.x <= 256) {  // a workgroup a unit: more under way in each
    ROWS_HALVES(4, 2, 2, 2)
  } else {  // (288 tiles of 3,584 of k at 4 / 8 / 12 rows 10.4 / 11.2 / 12.3 us, in batches of two steps 10.9 / 11.8 / 13.3)
    ROWS_HALVES(4, 1, 1, 1)
  }
#undef ROWS_HALVES
}

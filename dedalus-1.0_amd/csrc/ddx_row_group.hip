// Size-specialised plain x rows of batched plans whose members have an odd
// number of rows (pairs stay inside the member).  A unit of their own: beside
// the ungrouped kernels they moved the step's, instruction for instruction the
// same, to addresses where they share the instruction cache worse (512^2
// Boussinesq step 67.1 -> 68.4 us).
#include <hip/hip_runtime.h>

#include "ddx_fast.h"

namespace ddx {

template <typename T, int N, int V>
void row_group_go(hipStream_t s, const RowArgs<T>& a, long nrows, int group, dim3 grid) {
  if (a.mode == ROW_C2R) hipLaunchKernelGGL((row_c2r_fast<T, N, V, true>), grid, dim3(64), 0, s, a, nrows, group);
  else hipLaunchKernelGGL((row_r2c_fast<T, N, V, true>), grid, dim3(64), 0, s, a, nrows, group);
}

#define DDX_ROW_GROUP(T, N)                                                                     \
  template void row_group_go<T, N, 0>(hipStream_t, const RowArgs<T>&, long, int, dim3);         \
  template void row_group_go<T, N, 1>(hipStream_t, const RowArgs<T>&, long, int, dim3);
#define DDX_ROW_GROUPS(T) DDX_ROW_GROUP(T, 64) DDX_ROW_GROUP(T, 128) DDX_ROW_GROUP(T, 256) DDX_ROW_GROUP(T, 512)
DDX_ROW_GROUPS(double)
DDX_ROW_GROUPS(float)

}  // namespace ddx

// Batch decode kernel, dense launches over AWQ weights in groups of 64 rows (instantiations).
#include "q4_gemv_batch_launch.cuh"

namespace q4host {

void launch_batch_awq_g64(const BatchParams& bp, int dtype, int mt, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (dtype == Q4_DTYPE_F16) batch_rows_awq<Q4_DTYPE_F16, 64>(bp, mt, wk, fuse, grid, stream);
  else batch_rows_awq<Q4_DTYPE_BF16, 64>(bp, mt, wk, fuse, grid, stream);
}

}  // namespace q4host

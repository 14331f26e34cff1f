// Batch decode kernel, dense launches over AWQ weights in groups of 128 rows and more (instantiations).
#include "q4_gemv_batch_launch.cuh"

namespace q4host {

void launch_batch_awq(const BatchParams& bp, int dtype, int mt, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (dtype == Q4_DTYPE_F16) batch_rows_awq<Q4_DTYPE_F16, 128>(bp, mt, wk, fuse, grid, stream);
  else batch_rows_awq<Q4_DTYPE_BF16, 128>(bp, mt, wk, fuse, grid, stream);
}

}  // namespace q4host

// Batch decode kernel, dense launches over GPTQ weights in groups of 32 rows (instantiations).
#include "q4_gemv_batch_launch.cuh"

namespace q4host {

void launch_batch_gptq_g32(const BatchParams& bp, int dtype, int mt, int nq, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (dtype == Q4_DTYPE_F16) batch_rows_gptq<Q4_DTYPE_F16, 32>(bp, mt, nq, wk, fuse, grid, stream);
  else batch_rows_gptq<Q4_DTYPE_BF16, 32>(bp, mt, nq, wk, fuse, grid, stream);
}

}  // namespace q4host

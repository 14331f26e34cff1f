// Instantiations of the prefill kernels in q4_gemm_tall.cuh and q4_gemm_block.cuh: AWQ layout, fp16 activations.
#include "q4_gemm_block.cuh"
#include "q4_gemm_tall_launch.cuh"

namespace q4host {

void launch_tall_awq_f16(const q4::GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream) {
  launch_tall<Q4_DTYPE_F16, q4::kTileAwq>(gp, r, kw, fuse, grid, stream);
}

void launch_block_awq(const q4::GemmParams& gp, bool fuse, dim3 grid, hipStream_t stream) {
  auto k = fuse ? q4::gemm_block_kernel<q4::kTileAwq, true> : q4::gemm_block_kernel<q4::kTileAwq, false>;
  hipLaunchKernelGGL(k, grid, dim3(512), 0, stream, gp);
}

}  // namespace q4host

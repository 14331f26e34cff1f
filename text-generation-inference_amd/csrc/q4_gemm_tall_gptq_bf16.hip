// Instantiations of the prefill kernel in q4_gemm_tall.cuh: GPTQ layout, bf16 activations.
#include "q4_gemm_tall.cuh"
#include "q4_gemm_tall_launch.cuh"

namespace q4host {

void launch_tall_gptq_bf16(const q4::GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream) {
  launch_tall<Q4_DTYPE_BF16, q4::kTileGptq>(gp, r, kw, fuse, grid, stream);
}

}  // namespace q4host

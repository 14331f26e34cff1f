// Launch of one data type and layout of the prefill kernel in q4_gemm_tall.cuh (shared by the translation units
// that instantiate it).
#pragma once
#include "q4_gemm_tall.cuh"

namespace q4host {

template <int DTYPE, int LAYOUT, int R>
void launch_tall_rows(const q4::GemmParams& gp, int kw, bool fuse, dim3 grid, hipStream_t stream) {
  if constexpr (R <= 5 && LAYOUT == q4::kTileGptq) {
    if (kw == 2) {
      hipLaunchKernelGGL((q4::gemm_tall_kernel<DTYPE, LAYOUT, R, false, 2>), grid, dim3(256), 0, stream, gp);
      return;
    }
  }
  auto k = fuse ? q4::gemm_tall_kernel<DTYPE, LAYOUT, R, true> : q4::gemm_tall_kernel<DTYPE, LAYOUT, R, false>;
  hipLaunchKernelGGL(k, grid, dim3(256), 0, stream, gp);
}

template <int DTYPE, int LAYOUT>
void launch_tall(const q4::GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream) {
  switch (r) {
    case 3: return launch_tall_rows<DTYPE, LAYOUT, 3>(gp, kw, fuse, grid, stream);
    case 4: return launch_tall_rows<DTYPE, LAYOUT, 4>(gp, kw, fuse, grid, stream);
    case 5: return launch_tall_rows<DTYPE, LAYOUT, 5>(gp, kw, fuse, grid, stream);
    case 6: return launch_tall_rows<DTYPE, LAYOUT, 6>(gp, kw, fuse, grid, stream);
    default: return launch_tall_rows<DTYPE, LAYOUT, 8>(gp, kw, fuse, grid, stream);
  }
}

}  // namespace q4host

// Launches of the batch decode kernel, by layout and group length; the files that include this instantiate them.
#pragma once
#include "q4_gemv_batch.cuh"

namespace q4host {

using q4::BatchParams;

template <int DTYPE, int MT, int NQ, int WK, int GS>
static void batch_one_gptq(const BatchParams& bp, bool fuse, dim3 grid, hipStream_t stream) {
  using namespace q4;
  if (fuse) hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchGptq, MT, NQ, 1, WK, true, false, GS>), grid, dim3(64 * WK), 0, stream, bp);
  else hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchGptq, MT, NQ, 1, WK, false, false, GS>), grid, dim3(64 * WK), 0, stream, bp);
}

template <int DTYPE, int MT, int GS>
static void batch_tile_gptq(const BatchParams& bp, int nq, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (nq == 1 && wk == 8) batch_one_gptq<DTYPE, MT, 1, 8, GS>(bp, fuse, grid, stream);
  else if (nq == 1) batch_one_gptq<DTYPE, MT, 1, 4, GS>(bp, fuse, grid, stream);
  else if (wk == 8) batch_one_gptq<DTYPE, MT, 2, 8, GS>(bp, fuse, grid, stream);
  else batch_one_gptq<DTYPE, MT, 2, 4, GS>(bp, fuse, grid, stream);
}

// mt: blocks of 16 rows (1 to 4); nq: 64- or 128-column wave tiles; wk: 4 or 8 K waves
template <int DTYPE, int GS>
static void batch_rows_gptq(const BatchParams& bp, int mt, int nq, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (mt == 1) batch_tile_gptq<DTYPE, 1, GS>(bp, nq, wk, fuse, grid, stream);
  else if (mt == 2) batch_tile_gptq<DTYPE, 2, GS>(bp, nq, wk, fuse, grid, stream);
  else if (mt == 3) batch_tile_gptq<DTYPE, 3, GS>(bp, nq, wk, fuse, grid, stream);
  else batch_tile_gptq<DTYPE, 4, GS>(bp, nq, wk, fuse, grid, stream);
}

template <int DTYPE, int MT, int GS>
static void batch_tile_awq(const BatchParams& bp, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  using namespace q4;
  if (fuse) hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchAwq, MT, 2, 2, 4, true, false, GS>), grid, dim3(512), 0, stream, bp);
  else if (wk == 8) hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchAwq, MT, 2, 1, 8, false, false, GS>), grid, dim3(512), 0, stream, bp);
  else hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchAwq, MT, 2, 1, 4, false, false, GS>), grid, dim3(256), 0, stream, bp);
}

// mt: blocks of 16 rows (1 to 3); wk: 4 or 8 K waves (gated epilogue: 4 beside two column waves)
template <int DTYPE, int GS>
static void batch_rows_awq(const BatchParams& bp, int mt, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (mt == 1) batch_tile_awq<DTYPE, 1, GS>(bp, wk, fuse, grid, stream);
  else if (mt == 2) batch_tile_awq<DTYPE, 2, GS>(bp, wk, fuse, grid, stream);
  else batch_tile_awq<DTYPE, 3, GS>(bp, wk, fuse, grid, stream);
}

template <int DTYPE, int MT, int NQ, int WK, int GS>
static void batch_one_moe(const BatchParams& bp, bool fuse, dim3 grid, hipStream_t stream) {
  using namespace q4;
  if (fuse) hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchGptq, MT, NQ, 1, WK, true, true, GS>), grid, dim3(64 * WK), 0, stream, bp);
  else hipLaunchKernelGGL((gemv_batch_kernel<DTYPE, kBatchGptq, MT, NQ, 1, WK, false, true, GS>), grid, dim3(64 * WK), 0, stream, bp);
}

template <int DTYPE, int MT, int GS>
static void batch_tile_moe(const BatchParams& bp, int nq, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (nq == 1 && wk == 8) batch_one_moe<DTYPE, MT, 1, 8, GS>(bp, fuse, grid, stream);
  else if (nq == 1) batch_one_moe<DTYPE, MT, 1, 4, GS>(bp, fuse, grid, stream);
  else if (wk == 8) batch_one_moe<DTYPE, MT, 2, 8, GS>(bp, fuse, grid, stream);
  else batch_one_moe<DTYPE, MT, 2, 4, GS>(bp, fuse, grid, stream);
}

template <int DTYPE, int GS>
static void batch_rows_moe(const BatchParams& bp, int mt, int nq, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  if (mt == 1) batch_tile_moe<DTYPE, 1, GS>(bp, nq, wk, fuse, grid, stream);
  else if (mt == 2) batch_tile_moe<DTYPE, 2, GS>(bp, nq, wk, fuse, grid, stream);
  else if (mt == 3) batch_tile_moe<DTYPE, 3, GS>(bp, nq, wk, fuse, grid, stream);
  else batch_tile_moe<DTYPE, 4, GS>(bp, nq, wk, fuse, grid, stream);
}

}  // namespace q4host

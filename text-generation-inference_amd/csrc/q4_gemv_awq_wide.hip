// AWQ decode kernel for five to sixteen rows (q4_gemv_awq_wide.cuh): what it takes, its decomposition, and the launches.
#include "q4_gemv_awq_wide.cuh"

namespace q4host {

using q4::AwqFewParams;

// Decomposition: K waves and workgroups along K that minimise an estimate fitted to a sweep of 22 layer shapes x 5, 8 and 16 rows x
// both data types on MI355X (us): the 16 KB chunks that the waves of the busiest CU read, those that a wave walks one after the other in
// every round of resident workgroups (LDS: one of eight waves, two of four), the exchange levels and what they exchange (gate and
// up tiles: a level, half a plane).  Its picks are 1.7 % above the best measured ones on average, 12 % at worst.
static bool awq_wide_plan(const q4_weight* w, int M, bool gate_up, AwqFewPlan* plan) {
  const int chunks = w->K / 128;
  const long tiles = w->N / 256, plane = (long)w->N * M;  // sums that a split leaves
  double best = -1.0;
  for (int wk = 4; wk <= 8; wk += 4) {
    for (int sp = 1; sp <= 16 && wk * sp <= chunks; ++sp) {
      if ((sp - 1) * plane * 4 + (gate_up ? plane * 2 : 0) > Q4_WORKSPACE_CELL_BYTES) break;
      const long per_cu = (tiles * sp + 255) / 256, resident = 8 / wk, rounds = (tiles * sp + 256 * resident - 1) / (256 * resident);
      const int per_wave = (chunks + wk * sp - 1) / (wk * sp);
      double t = 0.46 * (double)(per_cu * wk) * per_wave + 0.8 * (double)rounds * per_wave + 3.8e-6 * ((sp - 1) + (gate_up ? 0.5 : 0.0)) * (double)plane;
      for (int cnt = sp; cnt > 1; cnt = (cnt + 1) >> 1) t += 0.55;
      if (best < 0.0 || t < best) {
        best = t;
        *plan = AwqFewPlan{1, wk, sp};
      }
    }
  }
  return best >= 0.0;
}

// Where this kernel is the one to run, against the batch decode kernel (64-byte pieces of the rows, half the K splits), which keeps
// what this one does not take: time of theirs over time of this one (48 shapes, 1.19 in geometric mean).
//   2^27 weights and more   1.18-1.48: 28672 x 8192, 16 rows 36.6 / 30.6 us, gated 8192 x 57344 79.3 / 57.0
//   8e7 to 2^27             1.06-1.33: 8192 x 10240, 5 rows 20.2 / 15.9, gated 4096 x 28672 16 rows 24.3 / 20.2, bf16 25.0 / 20.3
//   5e7 to 8e7              fp16 and gated up to 8 rows 1.00-1.27: 4096 x 12288 16 rows 13.6 / 12.2, 14336 x 4096 15.0 / 14.6, 18944 x
//                           3584 16.9 / 16.8; gated 9-16 rows 0.95-1.07 up to 6.1e7 (8320 x 6144 17.4 / 18.3), plain bf16 0.90-1.16
//                           (18944 x 3584 17.4 / 19.3): left out
//   less                    0.79-1.10: 11008 x 4096 13.4 / 14.8, 3584 x 8192 9.9 / 12.2, gated 2048 x 16384 11.3 / 12.0: many splits
//                           of few chunks, whose exchange outweighs the reads
bool awq_wide_default(const q4_weight* w, int M, int dtype, bool gate_up, AwqFewPlan* plan) {
  if (M <= q4::kAwqFewRows || M > q4::kAwqWideRows) return false;
  const long least = gate_up ? (M <= 8 ? 50000000 : 62000000) : (dtype == Q4_DTYPE_F16 ? 50000000 : 80000000);
  if ((long)w->K * w->N < least) return false;
  return awq_few_supported(w, M, gate_up) && awq_wide_plan(w, M, gate_up, plan);
}

template <int DTYPE>
static void launch_dtype(const AwqFewParams& p, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  using namespace q4;
  if (fuse && wk == 8) hipLaunchKernelGGL((gemv_awq_wide_kernel<DTYPE, 8, true>), grid, dim3(512), 0, stream, p);
  else if (fuse) hipLaunchKernelGGL((gemv_awq_wide_kernel<DTYPE, 4, true>), grid, dim3(256), 0, stream, p);
  else if (wk == 8) hipLaunchKernelGGL((gemv_awq_wide_kernel<DTYPE, 8, false>), grid, dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((gemv_awq_wide_kernel<DTYPE, 4, false>), grid, dim3(256), 0, stream, p);
}

void launch_awq_wide(const AwqFewParams& p, int dtype, const AwqFewPlan& plan, bool fuse, hipStream_t stream) {
  // (the meeting of gate and up tiles goes through the cells whatever the splits: the caller has seen to them)
  const dim3 grid((unsigned)(p.N / 256), (unsigned)p.splits);
  if (dtype == Q4_DTYPE_F16) launch_dtype<Q4_DTYPE_F16>(p, plan.wk, fuse, grid, stream);
  else launch_dtype<Q4_DTYPE_BF16>(p, plan.wk, fuse, grid, stream);
}

}  // namespace q4host

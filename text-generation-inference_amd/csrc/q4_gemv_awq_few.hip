// AWQ decode kernel for one to four rows (q4_gemv_awq_few.cuh): what it takes, its decomposition, and the launches (those of
// q4_gemv_awq_wide.cuh, which takes the same weights at more rows, go through here).
#include "q4_gemv_awq_few.cuh"

namespace q4host {

using q4::AwqFewParams;

void launch_awq_wide(const AwqFewParams& p, int dtype, const AwqFewPlan& plan, bool fuse, hipStream_t stream);

// Groups of 128 << s rows (or one group), K in whole 128-row chunks, N in whole wave tiles of 256 columns (gated epilogue: gate and
// up half each), tensors below 2 GB (32-bit offsets).
bool awq_few_supported(const q4_weight* w, int M, bool gate_up) {
  if (w->layout != Q4_LAYOUT_AWQ || M < 1) return false;
  if (w->K % 128 != 0 || w->K < 128 || w->N % (gate_up ? 512 : 256) != 0) return false;
  if (w->num_groups > 1) {
    const int per = w->groupsize / 128;
    if (w->groupsize % 128 != 0 || per < 1 || (per & (per - 1)) != 0) return false;
  }
  if ((long)w->num_groups * w->groupsize < w->K) return false;
  const long limit = 1L << 31;
  return (long)w->K * (w->N / 8) * 4 < limit && (long)w->num_groups * w->N * 2 < limit && (long)M * w->K * 2 < limit;
}

// Decomposition: column waves, K waves and workgroups along K that minimise an estimate fitted to a sweep of ten layer shapes on
// MI355X (us): the 16 KB chunks that the waves of the busiest CU read, those that a wave walks one after the
// other, and the exchange levels.
static bool awq_few_plan(const q4_weight* w, int M, bool gate_up, AwqFewPlan* plan) {
  const int chunks = w->K / 128;
  double best = -1.0;
  for (int wn = gate_up ? 2 : 1; wn <= 2; ++wn) {
    if (w->N % (256 * wn) != 0) continue;
    const long tiles = w->N / (256 * wn);
    for (int wk = 4; wk <= 8 / wn; wk += 4) {
      for (int sp = 1; sp <= 16 && wk * sp <= chunks; ++sp) {
        if ((long)(sp - 1) * w->N * M * 4 > Q4_WORKSPACE_CELL_BYTES) break;
        const long per_cu = (tiles * sp + 255) / 256;
        const int per_wave = (chunks + wk * sp - 1) / (wk * sp);
        double t = 0.58 * (double)(per_cu * wn * wk) * per_wave + 0.5 * per_wave + (per_cu > 1 ? 0.8 : 0.0);
        for (int cnt = sp; cnt > 1; cnt = (cnt + 1) >> 1) t += 0.45;
        if (best < 0.0 || t < best) {
          best = t;
          *plan = AwqFewPlan{wn, wk, sp};
        }
      }
    }
  }
  return best >= 0.0;
}

// Where this kernel is the one to run, against the words-as-stored kernel (gated: with the elementwise launch behind it) and the batch
// decode kernel that held the calls: 26 layer shapes x 1, 2 and 4 rows, time of theirs over time of this one, geometric mean (least).
//   plain fp16    1.22 (0.95: 2048 x 2048 at 4 rows 1.05); us, 14336 x 4096, 1 row 12.2 / 9.5, 8192 x 8192 13.0 / 9.5
//   plain bf16    1.19 (0.99)
//   gated fp16    1.25 (1.03); 4096 x 28672, 1 row 22.5 / 14.9
//   gated bf16    1.16 (1.03)
// Left to theirs: few rows of K, of which a wave walks one chunk in a long workgroup (plain below 2048: 1152 x 7168 0.84-0.91, 1024 x
// 8192 0.96-1.02; gated fp16 up to 1024: 1024 x 8192 0.95; gated bf16, 17 instead of nine operations a word to unpack, up to 2048:
// 2048 x 16384 0.97-0.99, 2048 x 2048 0.93); plain launches of 2^28 weights and more, which either reads at the copy rate (8192 x
// 57344 0.95-1.03).  So are layers of fewer 16 KB units (128 rows x 256 columns) than the chip has SIMDs, about 1000, of which some wave walks
// two: the CUs that have work then read twice what the batch kernel's 128-column tiles give them (chunks of K: us at one row, theirs / this one;
// 2122 calls of 14 widths x 22 lengths).
//   plain, up to 8192 rows of K   17 chunks x 4096 columns 0.91, bf16 0.85-0.86; 31 x 8192 bf16 0.90-0.93; fp16 from 600 units on (75 calls up to 1000,
//                                 weights from memory, 1.07, least 1.00: 47 x 5120 10.1 / 8.7; below, 194 calls 0.96), bf16 from 1000; longer ones 1.00 and more whatever the units
//   gated                         17 x 4096 0.81, 63 x 4096 0.89-0.92, 86 x 2048 0.93; fp16 from 1100 units on, bf16 from 1300, from 1000 beyond
//                                 8192 rows; 18 x 16384 0.92-0.95, bf16 0.89-0.90; weights from memory, 323 fp16 calls below the line 0.93
//   gated bf16, one chunk a wave  4096 x 4096 0.91-0.94, 4096 x 6144 0.98-1.00: from 800 units on
// (20480 columns in fp16 0.92-0.99 over 39-86 chunks, 19456 and 21504 1.1-1.3: kept.)
bool awq_few_default(const q4_weight* w, int M, int dtype, bool gate_up, AwqFewPlan* plan) {
  if (gate_up ? w->K <= (dtype == Q4_DTYPE_BF16 ? 2048 : 1024) : w->K < 2048 || (long)w->K * w->N >= (1L << 28)) return false;
  if (M > q4::kAwqFewRows || !awq_few_supported(w, M, gate_up)) return false;
  AwqFewPlan own;
  if (!awq_few_plan(w, M, gate_up, &own)) return false;
  const long chunks = w->K / 128, units = chunks * (w->N / 256);
  const bool bf16_gated = gate_up && dtype == Q4_DTYPE_BF16, one_each = chunks <= (long)own.wk * own.splits;
  if (!one_each && units < (w->K > 8192 ? (gate_up ? 1000 : 0) : (bf16_gated ? 1300 : (gate_up ? 1100 : (dtype == Q4_DTYPE_BF16 ? 1000 : 600))))) return false;
  if (bf16_gated && one_each && w->K <= 4096 && units < 800) return false;
  *plan = own;
  return true;
}

template <int DTYPE>
static void launch_dtype(const AwqFewParams& p, int wn, int wk, bool fuse, dim3 grid, hipStream_t stream) {
  using namespace q4;
  if (fuse) hipLaunchKernelGGL((gemv_awq_few_kernel<DTYPE, 2, 4, true>), grid, dim3(512), 0, stream, p);
  else if (wn == 2) hipLaunchKernelGGL((gemv_awq_few_kernel<DTYPE, 2, 4, false>), grid, dim3(512), 0, stream, p);
  else if (wk == 8) hipLaunchKernelGGL((gemv_awq_few_kernel<DTYPE, 1, 8, false>), grid, dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((gemv_awq_few_kernel<DTYPE, 1, 4, false>), grid, dim3(256), 0, stream, p);
}

int launch_awq_few(const q4_weight* w, const void* x, const void* bias, void* y, int M, int dtype, int gate_up_act, void* workspace,
                   size_t workspace_bytes, const AwqFewPlan& plan, hipStream_t stream) {
  const bool cells = workspace != nullptr && workspace_bytes >= Q4_WORKSPACE_COUNTER_BYTES;
  const int splits = cells ? plan.splits : 1;
  if (M > q4::kAwqFewRows && !cells) {
    set_error("q4_linear(AWQ, five to sixteen rows): a workspace of Q4_WORKSPACE_COUNTER_BYTES is needed");
    return Q4_ERR_WORKSPACE;
  }
  AwqFewParams p;
  p.qweight = w->qweight;
  p.qzeros = w->qzeros;
  p.scales = (const q4::half_t*)w->scales;
  p.x = x;
  p.bias = bias;
  p.y = y;
  p.cells = cells ? (unsigned long long*)((char*)workspace + Q4_WORKSPACE_TICKET_BYTES) : nullptr;
  p.N = w->N;
  p.K = w->K;
  p.M = M;
  p.cpw = w->K / 128 / (plan.wk * splits);
  p.rem = w->K / 128 % (plan.wk * splits);
  p.gshift = 31;
  if (w->num_groups > 1) {
    p.gshift = 0;
    while ((128 << p.gshift) < w->groupsize) ++p.gshift;
  }
  p.num_groups = w->num_groups;
  p.splits = splits;
  p.act = gate_up_act != 0 ? gate_up_act - 1 : 0;
  const dim3 grid((unsigned)(w->N / (256 * plan.wn)), (unsigned)splits);
  if (M > q4::kAwqFewRows) launch_awq_wide(p, dtype, plan, gate_up_act != 0, stream);
  else if (dtype == Q4_DTYPE_F16) launch_dtype<Q4_DTYPE_F16>(p, plan.wn, plan.wk, gate_up_act != 0, grid, stream);
  else launch_dtype<Q4_DTYPE_BF16>(p, plan.wn, plan.wk, gate_up_act != 0, grid, stream);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_linear(AWQ, %s rows): launch failed: %s", M > q4::kAwqFewRows ? "five to sixteen" : "up to four", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

}  // namespace q4host

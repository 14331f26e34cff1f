// Host side of the act-order batch decode kernel (q4_gemv_batch_act.cuh): what it takes, its decomposition, the launches.
#include "q4_gemv_batch_act.cuh"

namespace q4host {

using q4::BatchParams;

constexpr size_t kActLds = 160 * 1024 - 1024;  // of a workgroup

static int act_k_rows(const q4_weight* w, int wk, int splits) {  // largest K range of a workgroup
  const int chunks = w->K / 128, slots = wk * splits, cpw = chunks / slots, rem = chunks % slots;
  return (cpw * wk + (rem < wk ? rem : wk)) * 128;
}

// Up to four rows, four and more chunks a wave: x through LDS.  (Below, four steps in flight hold the table's loads back: 8192 x 8192, two
// chunks a wave, 12.8 us without and 13.0 with; 28672 x 8192, seven, 32.5 and 30.0.)
static bool act_few(const q4_weight* w, int M, int nq, int wk, int splits) {
  if (M > 4 || nq != 1 || w->K / 128 / (wk * splits) < 4) return false;
  // (not where the chunk's LDS costs a resident workgroup: 8192 x 57344 in groups of 32, whose two workgroups then just fill LDS, 72 us
  // without and 87 with)
  const size_t lds = kActLds, rows = act_k_rows(w, wk, splits);
  size_t resident = lds / q4::batch_act_lds(w->num_groups, (int)rows, wk, 1, 1, false);
  if (resident > (size_t)(16 / wk)) resident = 16 / wk;
  return lds / q4::batch_act_lds(w->num_groups, (int)rows, wk, 1, 1, true) >= resident;
}

// pair units of one exchange plane (see UNITS in q4_gemv_batch.cuh)
static long act_units(int nq, int M) { return nq == 2 ? M : (M + 1) / 2; }

static bool act_supported(const q4_weight* w, int M, bool gate_up) {
  if (w->g_idx == nullptr || w->layout != Q4_LAYOUT_GPTQ || M < 1 || w->K < 512 || w->K % 128 != 0 || w->N % (gate_up ? 128 : 64) != 0) return false;
  if (w->num_groups > 65535) return false;
  const long limit = 1L << 31;
  return (long)(w->K / 8) * w->N * 4 < limit && ((long)M + 64) * w->K * 2 < limit;
}

// Decomposition: K waves and K splits that minimise an estimate fitted to a sweep of 8 layer shapes x 6 row counts (1 to 64) on
// MI355X: the 128-row chunks a wave walks, alone and as one of the CU's waves, a further round of workgroups, their tables,
// the levels of the exchange and its traffic.  Its picks are 0.4 % above the best measured ones on average, 4.7 % at worst.
// uneven: the chunks that the busiest CU's waves walk over an even share.
// pow2: splits that are powers of two only.  Returns the estimate, or -1.
static double act_plan(const q4_weight* w, int M, int mt, bool pow2, BatchPlan* plan, double* uneven) {
  const int chunks = w->K / 128, tiles = w->N / 64;
  double best = -1.0;
  for (int wk = 8; wk >= 4; wk -= 4)
    for (int sp = 1; sp <= 16; sp += pow2 ? sp : 1) {
      if (wk * sp > chunks) break;
      if (sp > 1 && (long)(sp - 1) * act_units(1, M) * tiles * 512 > Q4_WORKSPACE_CELL_BYTES) break;
      const size_t lds = q4::batch_act_lds(w->num_groups, act_k_rows(w, wk, sp), wk, mt, 1, act_few(w, M, 1, wk, sp));
      if (lds > kActLds) continue;
      int resident = (int)(160 * 1024 / lds);
      const int by_registers = (mt <= 2 ? 16 : (mt == 3 ? 12 : 8)) / wk;
      if (resident > by_registers) resident = by_registers;
      const long wgs = (long)tiles * sp;
      const double per_wave = (double)((chunks + wk * sp - 1) / (wk * sp));
      const double per_cu = (double)((wgs + 255) / 256), rounds = (double)((wgs + 256L * resident - 1) / (256L * resident));
      double t = (0.653 + 0.229 * mt) * per_wave * (0.724 * rounds + 1.027 * per_cu * wk / 4.0) + 2.263 * (rounds - 1.0);
      t += 0.00334 * rounds * w->num_groups + 3.954e-6 * (sp - 1) * M * w->N;
      for (int s = sp; s > 1; s = (s + 1) >> 1) t += 0.392;
      if (best < 0.0 || t < best) {
        best = t;
        *plan = BatchPlan{1, wk, sp};
        *uneven = per_cu * wk * per_wave * 256.0 / ((double)chunks * tiles);
      }
    }
  return best;
}

// Gated fp16 launches up to 16 rows whose 128-column tiles fill the chip run on those: about one tile a CU as one round of eight
// waves, from one and a half on four waves, split along K as far as the cells allow (8192 x 57344, 4 rows, one
// workgroup / two / four along K: one zero point 53.3 / 54.0 / 53.7 us, others 67.8 / 67.1 / 65.1; on 64 columns 57-60 and 64-66).  In
// between (3584 x 37888, 296 tiles) a second round is nearly empty: 25.2 us, and 31.0 against 26.6 with several zero points.
// Below 5120 rows of K a workgroup along K has too few words to its table: from 384 tiles on 0.93-1.10 of the 64-column tiles' speed, 27 calls 0.98 in
// geometric mean (2304 x 50816 13 rows 23.6 us there, 25.4 here), from 5120 on 31 calls 1.06 (0.96-1.23), 192-256 tiles 1.06 (0.97-1.16).
static void act_wide(const q4_weight* w, int M, BatchPlan* plan) {
  const int chunks = w->K / 128, tiles = w->N / 128;
  if (w->N % 128 != 0 || tiles < 192 || (tiles > 256 && (tiles < 384 || w->K < 5120)) || w->num_groups > 96 || chunks < 16) return;
  int splits = 1;
  while (tiles > 256 && splits < 4 && (2L * splits - 1) * act_units(2, M) * tiles * 512 <= Q4_WORKSPACE_CELL_BYTES) splits *= 2;
  const int wk = tiles <= 256 ? 8 : 4;
  // (the table's rows are twice those that act_plan has seen to, and one workgroup along K holds the groups of all rows: K = 65536 stays on 64 columns)
  if (q4::batch_act_lds(w->num_groups, act_k_rows(w, wk, splits), wk, 1, 2, false) > kActLds) return;
  *plan = BatchPlan{2, wk, splits};
}

// Where this kernel runs, measured on MI355X against the kernels it takes over from (gemv_gptq_act_kernel in blocks of 16 rows
// up to 32, the MFMA kernel that unpacks into LDS from 33 on; gated: those and the elementwise kernel), 20 layer shapes, groups of
// 32 and 128, both types, time of theirs over time of this one in geometric mean (least):
//   1-5 rows 1.19 (0.96), 16 1.22 (1.00), 17 1.58 (1.07), 33 1.85 (1.35), 64 1.50 (1.15).  us, theirs / this one: 8192 x 57344
//   gated 1 row 85.7 / 67.8, 33 rows 205 / 123; 28672 x 8192 4 rows 41.8 / 36.7, 33 rows 125 / 54; 4096 x 4096 16 rows 9.5 / 7.7.
// K splits are powers of two unless the estimate of another number is a tenth below theirs, with two row blocks a fifth, and a fifth too
// where it gives up to sixteen rows four waves in place of eight: 293 such calls 1.13 in geometric mean over powers of two alone (0.93-1.48); 30 more of four
// waves for a tenth 0.99, 0.88 at worst (2560 x 10112 8 rows 9.5 / 10.8 us, 12800 x 18816 gated 5 bf16 rows 50.3 / 56.8).
// Plain launches of a few rows whose powers of two deal K out unevenly are the decode path's; up to five rows they run on this
// kernel all the same, with any number of splits (batch_act_few_default), us, gemv_gptq_act_kernel / so: 8192 x 10240, 4 rows 17.7 / 16.3,
// 9344 x 18560 40.5 / 27.9, 4096 x 11008 15.5 / 11.4, 3584 x 4608 8.2 / 7.5; 18 shapes 1.14 in geometric mean, one row of very long K
// 0.98 (18944 x 3584 15.4 / 15.7), left to the older kernel.  256 groups and more, whose tables leave room for fewer
// workgroups, among them: 8192 x 10240 in groups of 32, 1 row 20.1 / 20.1 (22.2 in powers of two), 4 rows 19.9 / 19.2, bf16 20.9 / 19.9 and 22.1 /
// 19.7; 94 calls of ten shapes, nearly all in groups of 32, 1.22 in geometric mean (1.00-1.78).  Left to the older kernel with such groups: 8192 x
// 10240 16 rows 22.4 / 23.3 (gated fp16 1 row 21.5 / 24.0, 16 rows 24.5 / 25.5, bf16 up to 2 rows; gated 9344 x 18560 is faster here, 1.1 and more), and 8192 x
// 57344 from 3 rows on, gated 5 rows 91.7 / 99.0.
bool batch_act_default(const q4_weight* w, int M, int dtype, bool gate_up, BatchPlan* plan) {
  double uneven = 1.0, uneven_any = 1.0;
  if (M > 64 || !act_supported(w, M, gate_up)) return false;
  const double pow2_us = act_plan(w, M, (M + 15) / 16, true, plan, &uneven);
  if (pow2_us < 0.0) return false;
  BatchPlan any;
  const double any_us = act_plan(w, M, (M + 15) / 16, false, &any, &uneven_any);
  if (any_us < ((M > 16 && M <= 32) || (M <= 16 && plan->wk == 8 && any.wk == 4) ? 0.8 : 0.9) * pow2_us) *plan = any;
  const double weights = (double)w->K * w->N;
  if (w->num_groups >= 256 && M <= 16 && weights >= 2.6e8 && M > 2) return false;
  if (w->num_groups >= 256 && M <= 16 && weights < 2.6e8 && uneven >= 1.19 && (!gate_up || (weights < 1.2e8 && (dtype == Q4_DTYPE_F16 || M <= 2))))
    return false;
  if (gate_up && dtype == Q4_DTYPE_F16 && M <= 16) act_wide(w, M, plan);
  if (gate_up || weights < 1.2e7) return true;
  if (w->groupsize < 64) return !(dtype == Q4_DTYPE_F16 && M <= 2 && uneven >= 1.9);
  return !(dtype == Q4_DTYPE_F16 ? M <= 5 && uneven >= 1.11 : M <= 2 && uneven >= 1.19 && w->K >= 8192);
}

// Plain calls of a few rows that batch_act_default leaves to the decode path (decode_few_default): with any number of workgroups along K.
bool batch_act_few_default(const q4_weight* w, int M, int dtype, BatchPlan* plan) {
  double uneven;
  if ((dtype == Q4_DTYPE_F16 && M == 1 && w->K > 5 * w->N) || (w->num_groups >= 256 && (double)w->K * w->N >= 2.6e8)) return false;
  return M <= 5 && act_supported(w, M, false) && act_plan(w, M, 1, false, plan, &uneven) >= 0.0;
}

static bool act_cells(const void* workspace, size_t workspace_bytes) {
  return workspace != nullptr && workspace_bytes >= Q4_WORKSPACE_COUNTER_BYTES;
}

// Without a workspace a workgroup walks all of K: the groups of all rows then have to lie in LDS beside the table.
bool batch_act_fits(const q4_weight* w, int M, const BatchPlan& plan, const void* workspace, size_t workspace_bytes) {
  return act_cells(workspace, workspace_bytes) || q4::batch_act_lds(w->num_groups, w->K, plan.wk, (M + 15) / 16, plan.nq, act_few(w, M, plan.nq, plan.wk, 1)) <= kActLds;
}

template <int DTYPE, int MT, int WK, bool FUSE, int NQ = 1, bool FEW = false>
static void act_one(const BatchParams& bp, dim3 grid, size_t lds, hipStream_t stream) {
  auto kernel = q4::gemv_batch_act_kernel<DTYPE, MT, WK, FUSE, NQ, FEW>;
  if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kernel, grid, dim3(64 * WK), lds, stream, bp);
}

template <int DTYPE, int MT>
static void act_tile(const BatchParams& bp, const BatchPlan& plan, bool fuse, bool few, dim3 grid, size_t lds, hipStream_t stream) {
  if constexpr (MT == 1) {
    if constexpr (DTYPE == Q4_DTYPE_F16) {
      if (plan.nq == 2) return (plan.wk == 8 ? act_one<DTYPE, 1, 8, true, 2> : act_one<DTYPE, 1, 4, true, 2>)(bp, grid, lds, stream);
    }
    if (few && plan.wk == 8) return (fuse ? act_one<DTYPE, 1, 8, true, 1, true> : act_one<DTYPE, 1, 8, false, 1, true>)(bp, grid, lds, stream);
    if (few) return (fuse ? act_one<DTYPE, 1, 4, true, 1, true> : act_one<DTYPE, 1, 4, false, 1, true>)(bp, grid, lds, stream);
  }
  if (plan.wk == 8) (fuse ? act_one<DTYPE, MT, 8, true> : act_one<DTYPE, MT, 8, false>)(bp, grid, lds, stream);
  else (fuse ? act_one<DTYPE, MT, 4, true> : act_one<DTYPE, MT, 4, false>)(bp, grid, lds, stream);
}

template <int DTYPE>
static void act_rows(const BatchParams& bp, int mt, const BatchPlan& plan, bool fuse, bool few, dim3 grid, size_t lds, hipStream_t stream) {
  if (mt == 1) act_tile<DTYPE, 1>(bp, plan, fuse, few, grid, lds, stream);
  else if (mt == 2) act_tile<DTYPE, 2>(bp, plan, fuse, few, grid, lds, stream);
  else if (mt == 3) act_tile<DTYPE, 3>(bp, plan, fuse, few, grid, lds, stream);
  else act_tile<DTYPE, 4>(bp, plan, fuse, few, grid, lds, stream);
}

int launch_batch_act(const q4_weight* w, const void* x, const void* bias, void* y, int M, int dtype, int gate_up_act, void* workspace,
                     size_t workspace_bytes, const BatchPlan& plan_in, hipStream_t stream) {
  BatchPlan plan = plan_in;
  const bool fuse = gate_up_act != 0;
  const int mt = (M + 15) / 16;
  if (plan.splits > 1 && !act_cells(workspace, workspace_bytes)) plan.splits = 1;
  // (a workgroup that walks all of K for want of a workspace holds the groups of all rows: on 64 columns where only that fits)
  if (plan.nq == 2 && q4::batch_act_lds(w->num_groups, act_k_rows(w, plan.wk, plan.splits), plan.wk, mt, 2, false) > kActLds) plan.nq = 1;
  const bool few = act_few(w, M, plan.nq, plan.wk, plan.splits);
  const size_t lds = q4::batch_act_lds(w->num_groups, act_k_rows(w, plan.wk, plan.splits), plan.wk, mt, plan.nq, few);
  if (lds > kActLds) {
    set_error("q4_linear(act-order batch kernel): %zu bytes of LDS needed%s", lds, act_cells(workspace, workspace_bytes) ? "" : " without a workspace");
    return Q4_ERR_WORKSPACE;
  }
  BatchParams bp = {};
  bp.qweight = w->qweight;
  bp.qzeros = w->qzeros;
  bp.scales = (const q4::half_t*)w->scales;
  bp.g_idx = w->g_idx;
  bp.x = x;
  bp.bias = bias;
  bp.y = y;
  bp.cells = plan.splits > 1 ? (unsigned long long*)((char*)workspace + Q4_WORKSPACE_TICKET_BYTES) : nullptr;
  bp.N = w->N;
  bp.K = w->K;
  bp.M = M;
  bp.x_rows = M;
  const int chunks = w->K / 128, slots = plan.wk * plan.splits;
  bp.cpw = chunks / slots;
  bp.rem = chunks % slots;
  bp.num_groups = w->num_groups;
  bp.splits = plan.splits;
  bp.units = (int)act_units(plan.nq, M);
  bp.act = fuse ? gate_up_act - 1 : 0;
  const dim3 grid((unsigned)(w->N / (64 * plan.nq)), (unsigned)plan.splits);
  if (dtype == Q4_DTYPE_F16) act_rows<Q4_DTYPE_F16>(bp, mt, plan, fuse, few, grid, lds, stream);
  else act_rows<Q4_DTYPE_BF16>(bp, mt, plan, fuse, few, grid, lds, stream);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_linear(act-order batch kernel): launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

}  // namespace q4host

// Host side of the prefill kernels in q4_gemm_tall.cuh and q4_gemm_block.cuh: what they take, where they are the faster
// ones, their plan, the launches.  The instantiations are in q4_gemm_tall_{gptq,awq}_{f16,bf16}.hip.
#include "q4_gemm_tall.cuh"

namespace q4host {

using q4::GemmParams;
using q4::Problem;

void launch_tall_gptq_f16(const GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream);
void launch_tall_gptq_bf16(const GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream);
void launch_tall_awq_f16(const GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream);
void launch_tall_awq_bf16(const GemmParams& gp, int r, int kw, bool fuse, dim3 grid, hipStream_t stream);
void launch_block_gptq(const GemmParams& gp, bool fuse, dim3 grid, hipStream_t stream);
void launch_block_awq(const GemmParams& gp, bool fuse, dim3 grid, hipStream_t stream);

bool gemm_tall_supported(const q4_weight* w, int M) {
  if (w->g_idx != nullptr || M < 1 || w->K < q4::kBK || w->K % q4::kBK != 0 || w->N % q4::kTallBN != 0) return false;
  if (w->groupsize < 64 || w->groupsize % 64 != 0 || (long)w->num_groups * w->groupsize < w->K) return false;
  // 32-bit byte offsets (x below 2 GB: rows past M lie past its end without wrapping)
  return ((long)M + 256) * w->K < (1L << 30) && (long)w->K * w->N < (1L << 32) && (long)w->num_groups * w->N < (1L << 30);
}

// us of one plan, as gemm_round_us: a K tile alone on the chip and with every CU at work (where the matrix pipes' power
// sets the pace), by layout, data type and tile height, the 256 x 256 kernel last.
static double tall_estimate_us(bool awq, int dtype, int M, int K, int N, int r, bool block, int splits) {
  static const double kTile[2][2][7][2] = {
      {{{0.62, 0.68}, {0.64, 0.90}, {0.74, 1.05}, {0.87, 1.22}, {0, 0}, {1.12, 1.61}, {1.32, 1.56}},
       {{0.71, 0.71}, {0.78, 0.96}, {0.86, 1.08}, {0.95, 1.21}, {0, 0}, {1.13, 1.56}, {0, 0}}},
      {{{0.94, 0.91}, {0.99, 1.12}, {1.04, 1.21}, {1.15, 1.38}, {0, 0}, {1.41, 1.76}, {1.37, 1.62}},
       {{1.06, 0.97}, {1.08, 1.20}, {1.17, 1.30}, {1.30, 1.47}, {0, 0}, {1.59, 1.82}, {0, 0}}}};
  const double* us = kTile[awq][dtype == Q4_DTYPE_BF16][block ? 6 : r - 3];
  const long tiles = (long)((M + 32 * r - 1) / (32 * r)) * (N / q4::kTallBN);
  const int KT = K / q4::kBK;
  const double t = gemm_round_us(tiles * splits, 256, (KT + splits - 1) / splits, us[0], us[1]);
  return t + 9.0 + (splits > 1 ? (double)splits * M * N * 8e-6 / 7.7 : 0.0);
}

// The plan with the smallest estimate.  K is split while the tiles alone leave CUs idle, at least four K tiles a
// workgroup, two rounds at most.  halves: K halves inside a workgroup too.
static double tall_plan(bool awq, int dtype, int M, int K, int N, bool gate_up, bool halves, TallPlan* plan) {
  static const int kSplits[] = {1, 2, 3, 4, 6, 8};
  double best = -1.0;
  for (int r = 3; r <= 9; ++r) {
    const bool block = r == 9;
    if (r == 7 || (block && dtype != Q4_DTYPE_F16)) continue;
    const int rr = block ? 8 : r;
    const long tiles = (long)((M + 32 * rr - 1) / (32 * rr)) * (N / q4::kTallBN);
    for (int sp : kSplits) {
      if (sp > 1 && (gate_up || tiles > 256 || tiles * sp > 512 || K / q4::kBK / sp < 4)) break;
      const double t = tall_estimate_us(awq, dtype, M, K, N, rr, block, sp);
      if (best < 0.0 || t < best) {
        best = t;
        *plan = TallPlan{rr, block, sp};
      }
    }
  }
  if (!halves || gate_up || awq || M > 1536) return best;
  // Two halves of K in a workgroup, 128 columns: as many CUs at work with half the splits, whose fp32 partial sums (8 M N bytes each, out and in)
  // otherwise cost up to a third of a call; every fragment of x then serves half as many columns, which is why they end where two
  // splits and less would do.  Fitted to 15 layer shapes x 100-640 rows x all heights and splits, within 7 % where the workgroups are one round;
  // where it puts them 2 % ahead they run.  1319 such calls at 65-1536 rows, weights from memory, 1.15 in geometric mean (0.93-1.77, 15 below
  // 0.97; 366 of serving models' layer shapes 1.12); us, before / so: 3584 x 8192 301 rows 33.9 / 28.9, bf16 35.2 / 30.3, 1024 x 8192 301 rows
  // 17.5 / 12.8, 14336 x 4096 89 rows 30.5 / 24.9, 3584 x 3584 1000 rows 39.9 / 34.3, 209 rows 19.7 / 21.1, 4096 x 6144 301 rows 29.9 / 29.6 (a whole
  // layer 0.995-1.00).  (A price on padded rows, which left the last two out, cost 90 calls that it changed 1.09 in geometric mean; a lead of 4 %
  // instead of 2 cost 534 calls 1.07.  AWQ, whose words are loaded row by row, 0.75-1.1: not built in.)
  static const double kHalves[3][2] = {{0.54, 0.81}, {0.69, 1.00}, {0.85, 1.23}};  // (bf16: 0.065 more)
  const int KT = K / q4::kBK;
  for (int r = 3; r <= 5; ++r)
    for (int sp : kSplits) {
      const long wgs = (long)((M + 32 * r - 1) / (32 * r)) * (N / (q4::kTallBN / 2)) * sp;
      if (KT % (2 * sp) != 0 || KT / (2 * sp) < 4 || wgs < 96 || wgs > 1024) continue;
      // A second round of workgroups starts and ends anew, which costs 4-6 us that the estimate does not know: below 4096 rows of K halves only
      // where all workgroups run at once (us, whole K ranges / halves in two rounds and more: 1024 x 16640 167 rows 18.1 / 23.4, 896 x 18944
      // 638 rows 30.3 / 42.9, 1152 x 17664 794 rows 48.7 / 57.6, 1792 x 43264 296 rows 68.0 / 74.3; 4096 x 45056 300 rows 140.9 / 142.2, 5632 x
      // 45056 258 rows 183.3 / 178.4, bf16 229.9 on 128-row workgroups / 180.9)
      if (wgs > 256 && K < 4096) continue;
      // (160-row tiles fill LDS and start late, which four or five K tiles a half don't make up for against 96-row tiles over whole K ranges: 640 x
      // 4864 825 rows 13.8 / 14.8, 640 x 10752 434 rows 14.4 / 15.3, 512 x 6144 679 rows 12.7 / 13.1; beyond 1024 rows those are left out below)
      if (r == 5 && K < 768 && M <= 1024) continue;
      const double more = dtype == Q4_DTYPE_BF16 ? 0.065 : 0.0;
      const double t = 1.02 * (gemm_round_us(wgs, 256, KT / (2 * sp), kHalves[r - 3][0] + more, kHalves[r - 3][1] + more) + 7.7 +
                               (sp > 1 ? 0.55 + 1.69e-6 * sp * M * N : 0.0));
      if (t < best) {
        best = t;
        *plan = TallPlan{r, false, sp, 2};
      }
    }
  return best;
}

// Where these kernels run: 8 % faster by estimate than the ones of q4_gemm.hip and q4_gemm_awq_direct.hip.  Measured
// on MI355X over 14 layer shapes (1024 x 8192 .. 28672 x 8192, gated 4096 x 28672, 3584 x 37888, 8192 x 57344) x
// 11 row counts (65 .. 2048), geometric mean of their time over the chosen kernel's: GPTQ fp16 1.07, bf16 1.08,
// AWQ fp16 1.05, bf16 1.04 (always the faster one: 1.10, 1.10, 1.07, 1.05); the tile heights and splits
// picked are 1 % above the best ones.  At 160 and 301 rows, where 128-row tiles pad most, 1.1-1.5.
// GPTQ gate_up projections of several rounds stay with the 128 x 256 tiles, two workgroups per CU (4096 x 28672 at
// 1400 rows 0.92-0.95, at 2048 0.92-0.99).
// The estimates are off by up to 15 %.  Over 19 layer shapes x 17 row counts (65 .. 2048) these kernels are the pick in 626
// cases: time of the others over theirs, geometric mean (least, most), GPTQ 1.13 (0.95, 1.55) in fp16, 1.16 (0.96, 1.60) in bf16,
// gated 1.20 (1.00, 1.58) and 1.17 (0.99, 1.52); AWQ 1.15 (0.97, 1.39), 1.17 (0.98, 1.34), gated 1.11 (0.97, 1.40) and 1.06
// (0.97, 1.26); the least is 8192 x 1280 at 512 rows.  What the estimates would give them beyond that, tall_outdone leaves to
// the others (the same quotient):
//   GPTQ, tiles below 256 rows, three rounds of the chip and more: every CU is at work, and these tiles unpack a weight as
//     often as two 128-row workgroups: 4096 x 28672 at 1400 and 2048 rows 0.93-0.96, 4096 x 12288 at 2048 0.92, gated 0.95,
//     8192 x 57344 at 1400 0.96; 256-row tiles in 3.5-7 rounds 0.97-1.06
//   GPTQ, 96-row tiles over whole K ranges for more than 1024 rows: 4096 x 4096 and 3584 x 3584 at 1400 0.93-0.94; at 700 0.97-1.07.  In K
//     halves, 128 columns wide, they are the faster ones, 30 calls 1.35 in geometric mean (1.00): 5120 x 2304 1040 rows 40.8 us on 128-row
//     workgroups, 38.9 so (42.5 on 160-row tiles in four splits), 6400 x 2048 1312 rows 54.6 / 46.4, 4096 x 2048 1245 bf16 rows 37.8 / 33.8
//   AWQ, K of 9 to 16 K tiles (shorter ones not measured), where start and epilogue count as much as the tiles in between: 1024 x 8192 at 1000
//     rows 0.90, gated bf16 at 512 to 1400 rows 0.86-1.02; up to 129 rows, in splits, 1.13-1.28, 256 x 256 tiles 1.20-1.34,
//     gated fp16 0.97-1.08
static bool tall_outdone(bool awq, int dtype, int M, int K, int N, bool gate_up, const TallPlan& plan) {
  if (plan.block) return false;
  if (awq) return K > 512 && K <= 1024 && M > 384 && (!gate_up || dtype == Q4_DTYPE_BF16);
  if (plan.kw == 2) return false;  // (128 columns: at most 512 tiles of 256, and 96 rows are no fault)
  const long tiles = (long)((M + 32 * plan.r - 1) / (32 * plan.r)) * (N / q4::kTallBN);
  return (plan.r < 8 && tiles >= 3 * 256) || (plan.r == 3 && !gate_up && M > 1024);
}

bool gemm_tall_default(const q4_weight* w, int M, int dtype, bool gate_up, TallPlan* plan) {
  if (M <= 64 || !gemm_tall_supported(w, M)) return false;
  const bool awq = w->layout == Q4_LAYOUT_AWQ;
  auto others = [&](bool fused) { return awq ? gemm_awq_direct_estimate_us(w, M, dtype) : gemm_estimate_us(w, M, fused); };
  auto taken = [&](double other) {
    return tall_plan(awq, dtype, M, w->K, w->N, gate_up, true, plan) * 1.08 < other && !tall_outdone(awq, dtype, M, w->K, w->N, gate_up, *plan);
  };
  if (!gate_up) return taken(others(false));
  const bool old_fused = gemm_gate_up_supported(w, M, dtype);
  if (old_fused && M > 1024 && (long)((M + 127) / 128) * (w->N / 256) > 1024) return false;
  double other = others(true);
  if (!old_fused) {
    // two launches: the faster plain kernel, the elementwise one
    TallPlan plain;
    const double t = tall_plan(awq, dtype, M, w->K, w->N, false, false, &plain);
    other = others(false);
    other = (t < other ? t : other) + 4.0 + (double)M * w->N * 3e-6 / 5.0;
  }
  return taken(other);
}

// fp32 partial tiles of the largest split any layout and data type would pick
size_t gemm_tall_workspace_bytes(int M, int K, int N) {
  if (M <= 64 || K < q4::kBK || K % q4::kBK != 0 || N % q4::kTallBN != 0) return 0;
  int splits = 1;
  for (int awq = 0; awq < 2; ++awq)
    for (int dtype : {Q4_DTYPE_F16, Q4_DTYPE_BF16}) {
      TallPlan plan;
      for (bool halves : {false, true}) {
        tall_plan(awq != 0, dtype, M, K, N, false, halves, &plan);
        if (plan.splits > splits) splits = plan.splits;
      }
    }
  return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

int launch_gemm_tall(const q4_weight* w, const void* x, const void* bias, void* y, int M, int dtype, int gate_up_act,
                     void* workspace, size_t workspace_bytes, const TallPlan& plan_in, hipStream_t stream) {
  TallPlan plan = plan_in;
  if (plan.splits > 1 && (workspace == nullptr || workspace_bytes < Q4_WORKSPACE_COUNTER_BYTES + (size_t)plan.splits * M * w->N * sizeof(float)))
    plan.splits = 1;
  GemmParams gp;
  gp.p = Problem{w->qweight, w->qzeros, (const q4::half_t*)w->scales, nullptr, x, bias, y,
                 M,          w->K,      w->N,                         w->groupsize, w->num_groups};
  gp.p.gate_up_act = gate_up_act;
  gp.moe = q4::MoeView{};
  gp.partial_rows = M;
  gp.splits = plan.splits;
  gp.partials = plan.splits > 1 ? (float*)((char*)workspace + Q4_WORKSPACE_COUNTER_BYTES) : nullptr;
  const int bm = 32 * plan.r;
  const long total = (long)((M + bm - 1) / bm) * (w->N / (q4::kTallBN / plan.kw)) * plan.splits;
  if (total > 0x7fffffffL) {
    set_error("q4_linear(gemm): grid too large");
    return Q4_ERR_UNSUPPORTED;
  }
  const dim3 grid((unsigned)total);
  const bool fuse = gate_up_act != 0, awq = w->layout == Q4_LAYOUT_AWQ;
  if (plan.block) (awq ? launch_block_awq : launch_block_gptq)(gp, fuse, grid, stream);
  else if (dtype == Q4_DTYPE_F16) (awq ? launch_tall_awq_f16 : launch_tall_gptq_f16)(gp, plan.r, plan.kw, fuse, grid, stream);
  else (awq ? launch_tall_awq_bf16 : launch_tall_gptq_bf16)(gp, plan.r, plan.kw, fuse, grid, stream);
  if (plan.splits > 1) launch_gemm_reduce(gp.partials, bias, y, M, w->N, plan.splits, dtype, stream);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_linear(gemm): launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

}  // namespace q4host

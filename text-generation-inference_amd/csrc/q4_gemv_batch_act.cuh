// Batch decode kernel for act-order weights (GPTQ layout with g_idx): y[M, N] = x @ dequant(W) for up to 64 activation rows,
// optionally with the gated-MLP epilogue.
//
// Every K row has its own group, so every weight looks its scale and zero point up: about four vector instructions a weight, which
// bound the launch (8192 x 57344 in fp16: the vector pipes issue two thirds of the time).  So:
//   * A weight is unpacked once for all rows; a further 16 rows cost four matrix instructions,
//     the fetch of their activations and four permutes per 32 x 64 weights.
//   * The table of scale | -(1024 + zero), one row of 64 columns per group, lies at the start of LDS and a row is 256 bytes: the
//     address of a lane's four columns is one byte permute of the group number and the lane's offset.
//   * A lane fetches the activations of its (row, K block) itself, 16 bytes a step from L2, ahead of the words that they
//     meet: LDS holds the table and the groups of the workgroup's K range, whatever the rows.
//   * K waves and K splits meet as in q4_gemv_batch.cuh.
// Measured on MI355X against gemv_gptq_act_kernel in blocks of 16 rows (gated: and the elementwise kernel), us: 28672 x 8192 16 rows
// 42.5 / 39.3, 17 rows 73.8 / 42.9; 8192 x 57344 gated 4 rows 86 / 67 (4 TB/s of packed weights); one layer of hidden size 8192
// at 4 rows, four projections, 155.8 / 133.2.
// With one zero point for all groups and columns of the tile (symmetric quantization) its permute drops out.
#pragma once
#include "q4_gemv_batch.cuh"

namespace q4 {

constexpr int kActTileBytes = 256;  // one group's row of the table
// LDS: table and groups, afterwards the sums of the K waves
constexpr size_t batch_act_lds(int num_groups, int k_rows, int wk, int mt) {
  const size_t table = (size_t)num_groups * kActTileBytes + (size_t)k_rows * 2, sums = (size_t)wk * mt * 4096;
  return table > sums ? table : sums;
}

template <int DTYPE, int MT, int WK, bool FUSE>
__global__ __launch_bounds__(64 * WK, MT <= 2 ? 4 : (MT == 3 ? 3 : 2)) void gemv_batch_act_kernel(BatchParams bp) {
  extern __shared__ __align__(16) unsigned char act_lds[];
  constexpr int PF = 2;  // 32-row steps in flight
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kq = lane >> 4;
  const int N = bp.N, half = N >> 1, tile = blockIdx.x;
  const int split = blockIdx.y, M = bp.M;
  const int col = FUSE ? tile * 32 + 4 * (j & 7) + (j >> 3) * half : tile * 64 + 4 * j;

  const int slot0 = split * WK, slot = slot0 + wave;
  auto first_chunk = [&](int s) { return s * bp.cpw + min(s, bp.rem); };
  const int wg0 = first_chunk(slot0) * 128, wg_rows = first_chunk(slot0 + WK) * 128 - wg0;
  const int k0 = first_chunk(slot) * 128;
  const int nsteps = (first_chunk(slot + 1) * 128 - k0) / 32;  // four and more, even

  const direct_rsrc_t wrsrc = direct_rsrc(bp.qweight, (uint32_t)(bp.K >> 3) * (uint32_t)N * 4u);
  const direct_rsrc_t xrsrc = direct_rsrc(bp.x, (uint32_t)bp.x_rows * (uint32_t)bp.K * 2u);
  const uint32_t w_lane = ((uint32_t)kq * (uint32_t)N + (uint32_t)col) * 4u;
  uint32_t x_lane[MT];  // rows past the end lie past the end of x: zeros, no memory touched
#pragma unroll
  for (int m = 0; m < MT; ++m) x_lane[m] = ((uint32_t)(16 * m + j) * (uint32_t)bp.K + (uint32_t)kq * 8u) * 2u;
  struct Step {
    uint4_t x[MT], w;
  };
  auto load_step = [&](int st, Step& s) {
    const uint32_t k = scalar_u32((uint32_t)(k0 + st * 32));
#pragma unroll
    for (int m = 0; m < MT; ++m) s.x[m] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, x_lane[m], k * 2u, 0));
    s.w = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, w_lane, (k >> 3) * (uint32_t)N * 4u, 2));
  };
  Step ring[PF];
#pragma unroll
  for (int b = 0; b < PF; ++b) load_step(b, ring[b]);

  // ---- groups of the workgroup's K rows, clamped to the table, as 16 bits; four loads of a thread in flight
  constexpr int PU = 4;
  constexpr int THREADS = 64 * WK;
  const int tid = threadIdx.x;
  uint16_t* groups = (uint16_t*)(act_lds + (size_t)bp.num_groups * kActTileBytes);
  {
    const int32_t* src = bp.g_idx + wg0;
    const int quads = wg_rows >> 2, gmax = bp.num_groups - 1;
    for (int i0 = tid; i0 < quads; i0 += PU * THREADS) {
      uint4_t v[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u)
        if (i0 + u * THREADS < quads) v[u] = *(const uint4_t*)(src + 4 * (i0 + u * THREADS));
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        if (i0 + u * THREADS >= quads) continue;
        uint32_t g[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) g[q] = (uint32_t)min(max((int)v[u][q], 0), gmax);
        *(uint2_t*)(groups + 4 * (i0 + u * THREADS)) = uint2_t{g[0] | (g[1] << 16), g[2] | (g[3] << 16)};
      }
    }
  }
  // ---- table: scale | -(1024 + zero) << 16 of the tile's 64 columns (gated epilogue: 32 gate, 32 up), all groups
  uint32_t zref, zdiff;
  {
    auto octet = [&](int c8) { return FUSE ? tile * 32 + 8 * (c8 & 3) + (c8 >> 2) * half : tile * 64 + 8 * c8; };
    const int items = bp.num_groups * 8;
    zref = gptq_zero_plus_one(bp.qzeros[octet(0) >> 3]);
    zdiff = zref ^ ((zref & 0xFu) * 0x11111111u);
    for (int i0 = tid; i0 < items; i0 += PU * THREADS) {
      uint32_t zr[PU];
      uint4_t sr[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int i = i0 + u * THREADS;
        if (i < items) {
          const int n = octet(i & 7);
          zr[u] = bp.qzeros[(size_t)(i >> 3) * (N >> 3) + (n >> 3)];
          sr[u] = *(const uint4_t*)(bp.scales + (size_t)(i >> 3) * N + n);
        }
      }
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int i = i0 + u * THREADS;
        if (i >= items) continue;
        const uint32_t z8 = gptq_zero_plus_one(zr[u]);
        zdiff |= z8 ^ zref;
        uint32_t e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const uint32_t s16 = (q & 1) ? (sr[u][q >> 1] >> 16) : (sr[u][q >> 1] & 0xFFFFu);
          e[q] = s16 | ((0xE400u | ((z8 >> (4 * q)) & 0xFu)) << 16);
        }
        uint4_t* dst = (uint4_t*)(act_lds + (size_t)i * 32);
        dst[0] = uint4_t{e[0], e[1], e[2], e[3]};
        dst[1] = uint4_t{e[4], e[5], e[6], e[7]};
      }
    }
  }
  const bool one_zero = __syncthreads_or((int)(zdiff != 0u)) == 0;
  const uint32_t c_const = 0xE400E400u | (zref & 0xFu) | ((zref & 0xFu) << 16);

  const uint16_t* g_lane = groups + (k0 - wg0) + kq * 8;
  const uint32_t lane16 = (uint32_t)j * 16u;  // the lane's four columns in a row of the table
  const SpliceConsts splice = splice_consts();
  float4_t acc[4][MT];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = float4_t{0.f, 0.f, 0.f, 0.f};

  auto process = [&](int st, const Step& s, auto one_zero_c) __attribute__((always_inline)) {
    constexpr bool ONE_ZERO = decltype(one_zero_c)::value;
    uint4_t a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {  // K order [0,4,1,5,2,6,3,7] of the splice
      a[m].x = __builtin_amdgcn_perm(s.x[m].z, s.x[m].x, 0x05040100u);
      a[m].y = __builtin_amdgcn_perm(s.x[m].z, s.x[m].x, 0x07060302u);
      a[m].z = __builtin_amdgcn_perm(s.x[m].w, s.x[m].y, 0x05040100u);
      a[m].w = __builtin_amdgcn_perm(s.x[m].w, s.x[m].y, 0x07060302u);
    }
    const uint4_t g8 = *(const uint4_t*)(g_lane + st * 32);
    uint4_t e[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) e[r] = *(const uint4_t*)(act_lds + __builtin_amdgcn_perm(g8[r >> 1], lane16, (r & 1) ? 0x0C070600u : 0x0C050400u));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint4_t b;
#pragma unroll
      for (int pr = 0; pr < 4; ++pr) {
        // rows pr and pr + 4 of the K block share one splice (nibbles 16 bits apart)
        const uint32_t ea = e[pr][t], eb = e[pr + 4][t];
        const uint32_t c2 = ONE_ZERO ? c_const : __builtin_amdgcn_perm(eb, ea, 0x07060302u);
        const uint32_t q2 = ((s.w[t] >> (4 * pr)) & splice.mask_lo) | splice.magic;
        const half2_t dq = as_half2(q2) + as_half2(c2);  // exact q - z
        if constexpr (DTYPE == Q4_DTYPE_F16) {
          b[pr] = as_u32(dq * as_half2(__builtin_amdgcn_perm(eb, ea, 0x05040100u)));  // one fp16 rounding, as the reference
        } else {
          // the exact fp32 products from the fp16 halves where they lie, rounded once by the packed convert
          const uint32_t dqu = as_u32(dq);
          float2_t f;
          asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,1,0]" : "=v"(f.x) : "v"(dqu), "v"(ea));
          asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,1,0]" : "=v"(f.y) : "v"(dqu), "v"(eb));
          b[pr] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, gemm_bf16x2_t));
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) batch_mfma<DTYPE>(a[m], b, acc[t][m]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto walk = [&](auto one_zero_c) __attribute__((always_inline)) {
    for (int st = 0; st < nsteps - PF; st += PF) {
#pragma unroll
      for (int b = 0; b < PF; ++b) {
        process(st + b, ring[b], one_zero_c);
        load_step(st + b + PF, ring[b]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int b = 0; b < PF; ++b) process(nsteps - PF + b, ring[b], one_zero_c);
  };
  if (one_zero) walk(std::true_type{});
  else walk(std::false_type{});

  __syncthreads();  // everybody is done with the table
  auto sums = [&](int w, int m, int r) { return (float*)(act_lds + (size_t)(w * MT + m) * 4096 + r * 256); };
  batch_finish<DTYPE, false, MT, 1, 1, WK, FUSE, false>(bp, acc, sums, lane, wave, tile, split, 0, 0, M);
}

}  // namespace q4

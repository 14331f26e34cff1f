// Batch decode kernel for act-order weights (GPTQ layout with g_idx): y[M, N] = x @ dequant(W) for up to 64 activation rows,
// optionally with the gated-MLP epilogue.
//
// Every K row has its own group, so every weight looks its scale and zero point up: about four vector instructions a weight, which
// bound the launch (8192 x 57344 in fp16: the vector pipes issue two thirds of the time).  So:
//   * A weight is unpacked once for all rows; a further 16 rows cost four matrix instructions,
//     the fetch of their activations and four permutes per 32 x 64 weights.
//   * The table, per group and four columns their scales and -(1024 + zero), lies at the start of LDS and a row of it is 256 or 512
//     bytes: the address of a lane's columns is one byte permute of the group number and the lane's offset.
//   * With one zero point for all groups and columns of the tile (symmetric quantization) only scales are looked up, half the
//     bytes, and the splices of odd nibbles need no shift.
//   * A lane fetches the activations of its (row, K block) itself, 16 bytes a step from L2, ahead of the words that they
//     meet: LDS holds the table and the groups of the workgroup's K range, whatever the rows.  Up to four rows (FEW) one
//     load fetches a 128-row chunk of all of them, which a wave passes through 1 KB of LDS: three of four such loads were for rows
//     that are not there (28672 x 8192, 4 rows 32.5 us, so 30.0).
//   * NQ = 2, gated epilogue: a wave owns 64 gate and 64 up columns instead of 32 and 32.  It then reads 256 bytes of a row in one piece;
//     in two of 128 the same launch, without any arithmetic, takes 50 us on 8192 x 57344, in pieces of 256 bytes 40.
//   * K waves and K splits meet as in q4_gemv_batch.cuh.
// Measured on MI355X against gemv_gptq_act_kernel in blocks of 16 rows (gated: and the elementwise kernel), us: 28672 x 8192 16 rows
// 42.5 / 39.3, 17 rows 73.8 / 42.9; 8192 x 57344 gated 4 rows 86 / 67 (4 TB/s of packed weights); one layer of hidden size 8192
// at 4 rows, four projections, 155.8 / 133.2.
#pragma once
#include "q4_gemv_batch.cuh"
#include "q4_gemv_lean.cuh"

namespace q4 {

// LDS: table, groups and (few rows) a chunk of x per wave, afterwards the sums of the K waves
constexpr size_t batch_act_lds(int num_groups, int k_rows, int wk, int mt, int nq, bool few) {
  const size_t table = (size_t)num_groups * (nq * 256) + (size_t)k_rows * 2 + (few ? wk * 1024 : 0), sums = (size_t)wk * mt * 4096;
  return table > sums ? table : sums;
}

// NQ: quads of columns of a lane, 64 NQ columns a wave (2: gated epilogue).  FEW: up to four rows.
template <int DTYPE, int MT, int WK, bool FUSE, int NQ, bool FEW>
__global__ __launch_bounds__(64 * WK, NQ == 2 ? 2 : (MT <= 2 ? 4 : (MT == 3 ? 3 : 2))) void gemv_batch_act_kernel(BatchParams bp) {
  static_assert(NQ == 1 || (NQ == 2 && FUSE && MT == 1), "128-column tiles: gated epilogue, one row block");
  static_assert(!FEW || (MT == 1 && NQ == 1), "few rows are one row block");
  extern __shared__ __align__(16) unsigned char act_lds[];
  constexpr int PF = FEW ? 4 : 2;  // 32-row steps in flight (FEW: a chunk)
  constexpr int F = 4 * NQ;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kq = lane >> 4;
  const int N = bp.N, half = N >> 1, tile = blockIdx.x;
  const int split = blockIdx.y, M = bp.M;
  const int col = FUSE && NQ == 1 ? tile * 32 + 4 * (j & 7) + (j >> 3) * half : tile * 64 + 4 * j;  // NQ = 2: and half + col

  const int slot0 = split * WK, slot = slot0 + wave;
  auto first_chunk = [&](int s) { return s * bp.cpw + min(s, bp.rem); };
  const int wg0 = first_chunk(slot0) * 128, wg_rows = first_chunk(slot0 + WK) * 128 - wg0;
  const int k0 = first_chunk(slot) * 128;
  const int nsteps = (first_chunk(slot + 1) * 128 - k0) / 32;  // four and more, a multiple of four

  const direct_rsrc_t wrsrc = direct_rsrc(bp.qweight, (uint32_t)(bp.K >> 3) * (uint32_t)N * 4u);
  const direct_rsrc_t xrsrc = direct_rsrc(bp.x, (uint32_t)bp.x_rows * (uint32_t)bp.K * 2u);
  const uint32_t w_lane = ((uint32_t)kq * (uint32_t)N + (uint32_t)col) * 4u;
  // rows past the end lie past the end of x: zeros, no memory touched.  FEW: lane l fetches row l / 16, bytes 16 (l % 16) ..
  // of a chunk's 256
  uint32_t x_lane[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    x_lane[m] = FEW ? ((uint32_t)kq * (uint32_t)bp.K + (uint32_t)j * 8u) * 2u : ((uint32_t)(16 * m + j) * (uint32_t)bp.K + (uint32_t)kq * 8u) * 2u;
  struct Step {
    uint4_t x[FEW ? 1 : MT], w[NQ];
  };
  auto load_x = [&](int st, uint4_t (&x)[FEW ? 1 : MT]) __attribute__((always_inline)) {
    const uint32_t k = scalar_u32((uint32_t)(k0 + st * 32));
#pragma unroll
    for (int m = 0; m < MT; ++m) x[m] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, x_lane[m], k * 2u, 0));
  };
  auto load_step = [&](int st, Step& s) __attribute__((always_inline)) {
    if constexpr (!FEW) load_x(st, s.x);
    const uint32_t k = scalar_u32((uint32_t)(k0 + st * 32));
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      s.w[q] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, w_lane, ((k >> 3) * (uint32_t)N + q * (uint32_t)half) * 4u, 2));
  };
  Step ring[PF];
  uint4_t x_chunk[FEW ? 1 : MT];  // FEW: of the next chunk
  if constexpr (FEW) load_x(0, x_chunk);
#pragma unroll
  for (int b = 0; b < PF; ++b) load_step(b, ring[b]);

  // ---- groups of the workgroup's K rows, clamped to the table, as 16 bits; four loads of a thread in flight
  constexpr int PU = 4;
  constexpr int THREADS = 64 * WK;
  const int tid = threadIdx.x;
  constexpr int ROW = 256 * NQ;  // bytes of the table per group
  uint16_t* groups = (uint16_t*)(act_lds + (size_t)bp.num_groups * ROW);  // 256-byte pieces before the row's group
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
        for (int q = 0; q < 4; ++q) g[q] = (uint32_t)min(max((int)v[u][q], 0), gmax) * NQ;
        *(uint2_t*)(groups + 4 * (i0 + u * THREADS)) = uint2_t{g[0] | (g[1] << 16), g[2] | (g[3] << 16)};
      }
    }
  }
  // ---- table: four scales and four -(1024 + zero) per column quad of the tile (gated epilogue: gate, then up), all groups
  uint32_t zref, zdiff;
  {
    constexpr int OCT = 8 * NQ;  // columns in eights
    auto octet = [&](int c8) { return FUSE ? tile * (32 * NQ) + 8 * (c8 & (OCT / 2 - 1)) + (c8 / (OCT / 2)) * half : tile * 64 + 8 * c8; };
    const int items = bp.num_groups * OCT;
    zref = gptq_zero_plus_one(bp.qzeros[octet(0) >> 3]);
    zdiff = zref ^ ((zref & 0xFu) * 0x11111111u);
    for (int i0 = tid; i0 < items; i0 += PU * THREADS) {
      uint32_t zr[PU];
      uint4_t sr[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int i = i0 + u * THREADS;
        if (i < items) {
          const int n = octet(i % OCT);
          zr[u] = bp.qzeros[(size_t)(i / OCT) * (N >> 3) + (n >> 3)];
          sr[u] = *(const uint4_t*)(bp.scales + (size_t)(i / OCT) * N + n);
        }
      }
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int i = i0 + u * THREADS;
        if (i >= items) continue;
        const uint32_t z8 = gptq_zero_plus_one(zr[u]);
        zdiff |= z8 ^ zref;
        uint32_t z2[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) z2[q] = 0xE400E400u | ((z8 >> (8 * q)) & 0xFu) | (((z8 >> (8 * q + 4)) & 0xFu) << 16);
        uint4_t* const dst = (uint4_t*)(act_lds + (size_t)i * 32);
        dst[0] = uint4_t{sr[u][0], sr[u][1], z2[0], z2[1]};
        dst[1] = uint4_t{sr[u][2], sr[u][3], z2[2], z2[3]};
      }
    }
  }
  const bool one_zero = __syncthreads_or((int)(zdiff != 0u)) == 0;
  // -(1024 + zero), -(64 + zero) of the one zero point
  const uint32_t c_low = 0xE400E400u | (zref & 0xFu) | ((zref & 0xFu) << 16), c_high = 0xD400D400u | ((zref & 0xFu) << 4) | ((zref & 0xFu) << 20);

  const uint16_t* g_lane = groups + (k0 - wg0) + kq * 8;
  unsigned char* const xbuf = (unsigned char*)(groups + wg_rows) + wave * 1024;  // FEW: this wave's chunk of x
  const uint32_t lane16 = (uint32_t)j * 16u;  // the lane's four columns in a row of the table
  const LeanConsts splice = lean_consts<Q4_DTYPE_F16>();
  float4_t acc[F][MT];
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[f][m] = float4_t{0.f, 0.f, 0.f, 0.f};
  // 16 bytes of x into the K order [0,4,1,5,2,6,3,7] of the splice
  auto k_order = [](const uint4_t v) __attribute__((always_inline)) {
    return uint4_t{__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                   __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
  };

  auto process = [&](int st, const Step& s, auto one_zero_c) __attribute__((always_inline)) {
    constexpr bool ONE_ZERO = decltype(one_zero_c)::value;
    uint4_t a[MT];
    if constexpr (FEW) {
      a[0] = *(const uint4_t*)(xbuf + (j & 3) * 256 + (st & 3) * 64 + kq * 16);
    } else {
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = k_order(s.x[m]);
    }
    const uint4_t g8 = *(const uint4_t*)(g_lane + st * 32);
    uint2_t es[8][NQ], ez[8][NQ];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const unsigned char* const at = act_lds + __builtin_amdgcn_perm(g8[r >> 1], lane16, (r & 1) ? 0x0C070600u : 0x0C050400u);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if constexpr (ONE_ZERO) {
          es[r][q] = *(const uint2_t*)(at + q * 256);
        } else {
          const uint4_t e = *(const uint4_t*)(at + q * 256);
          es[r][q] = uint2_t{e.x, e.y};
          ez[r][q] = uint2_t{e.z, e.w};
        }
      }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u;  // a column's half of two registers side by side
      const int q = f / 4, t = f % 4;
      const uint32_t w = s.w[q][t], w8 = w >> 8, sel = (t & 1) ? kHigh : kLow;
      uint4_t b;
#pragma unroll
      for (int pr = 0; pr < 4; ++pr) {
        // rows pr and pr + 4 of the K block share one splice (nibbles 16 bits apart)
        const uint32_t ea = t < 2 ? es[pr][q].x : es[pr][q].y, eb = t < 2 ? es[pr + 4][q].x : es[pr + 4][q].y;
        half2_t dq;  // exact q - z
        if constexpr (ONE_ZERO) {
          const uint32_t v = pr < 2 ? w : w8;
          dq = (pr & 1) ? as_half2((v & splice.mask_hi) | splice.magic_hi) + as_half2(c_high) : as_half2((v & splice.mask_lo) | splice.magic_lo) + as_half2(c_low);
        } else {
          const uint32_t za = t < 2 ? ez[pr][q].x : ez[pr][q].y, zb = t < 2 ? ez[pr + 4][q].x : ez[pr + 4][q].y;
          dq = as_half2(((w >> (4 * pr)) & splice.mask_lo) | splice.magic_lo) + as_half2(__builtin_amdgcn_perm(zb, za, sel));
        }
        if constexpr (DTYPE == Q4_DTYPE_F16) {
          b[pr] = as_u32(dq * as_half2(__builtin_amdgcn_perm(eb, ea, sel)));  // one fp16 rounding, as the reference
        } else {
          // the exact fp32 products from the fp16 halves where they lie, rounded once by the packed convert
          const uint32_t dqu = as_u32(dq);
          float2_t v;
          if (t & 1) {
            asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[1,1,0]" : "=v"(v.x) : "v"(dqu), "v"(ea));
            asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(v.y) : "v"(dqu), "v"(eb));
          } else {
            asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,1,0]" : "=v"(v.x) : "v"(dqu), "v"(ea));
            asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,1,0]" : "=v"(v.y) : "v"(dqu), "v"(eb));
          }
          b[pr] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, gemm_bf16x2_t));
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) batch_mfma<DTYPE>(a[m], b, acc[f][m]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto walk = [&](auto one_zero_c) __attribute__((always_inline)) {
    // (the x of a chunk goes through LDS when its first step is due: the wave's reads of the chunk before are in order ahead)
    auto chunk_x = [&](int st, bool more) __attribute__((always_inline)) {
      if constexpr (FEW) {
        *(uint4_t*)(xbuf + lane * 16) = k_order(x_chunk[0]);
        if (more) load_x(st + PF, x_chunk);
      }
    };
    for (int st = 0; st < nsteps - PF; st += PF) {
      chunk_x(st, true);
#pragma unroll
      for (int b = 0; b < PF; ++b) {
        process(st + b, ring[b], one_zero_c);
        load_step(st + b + PF, ring[b]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    chunk_x(nsteps - PF, false);
#pragma unroll
    for (int b = 0; b < PF; ++b) process(nsteps - PF + b, ring[b], one_zero_c);
  };
  if (one_zero) walk(std::true_type{});
  else walk(std::false_type{});

  __syncthreads();  // everybody is done with the table
  auto sums = [&](int w, int m, int r) { return (float*)(act_lds + (size_t)(w * MT + m) * 4096 + r * 256); };
  batch_finish<DTYPE, false, MT, NQ, 1, WK, FUSE, false>(bp, acc, sums, lane, wave, tile, split, 0, 0, M);
}

}  // namespace q4

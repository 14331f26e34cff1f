// Decode kernel for the AWQ layout (qweight [K, N/8]: a word holds eight interleaved columns of one K row), five to sixteen activation
// rows, optionally with the gated-MLP epilogue.
//
// What bounds it is the stream of packed words, as in q4_gemv_awq_few.cuh, and so the wave tile is the same: 256 columns, two words a
// lane, whole 128-byte lines of every row (the batch kernel's 128-column tiles read 64-byte pieces, at 60-70 % of the rate).  With more
// rows than four the words are put into K order:
//   * Bytes of two K rows side by side, the splice and the zero point's subtraction give pairs of exact integers q - z, ten vector
//     instructions a word; one 16x16x32 MFMA then serves sixteen rows, where words as stored take four.
//   * The scale multiplies the fp32 sum of a 128-row chunk, which lies inside one group; both sets of sums, 128 registers, fit
//     two waves a SIMD for one row block only.
//   * x goes from L2 into LDS without registers, 64 K rows of a wave at a time, XORed as in q4_gemv_batch.cuh; no barrier before the K
//     waves meet.
//   * Tiles are few and K splits many, and what they exchange grows with the rows: a workgroup is one tile of K waves, and with the gated
//     epilogue a gate tile and its up tile are two workgroups that meet in one more exchange (as one workgroup they would cost twice
//     the K splits, which the exchange cells do not hold at 16 rows of 4096 x 28672).
// Measured on MI355X against the batch kernel, us: gated 4096 x 28672, 5 rows 22.3 / 17.9, 16 rows 24.3 / 20.2 (a kernel that only reads
// takes 13.0 on this grid, in 64-byte pieces 22); 28672 x 8192, 16 rows 36.6 / 29.4.
#pragma once
#include "q4_gemv_awq_few.cuh"
#include "q4_gemv_batch.cuh"

namespace q4 {

constexpr int kAwqWideRows = 16;

// WK: K waves.
template <int DTYPE, int WK, bool FUSE>
__global__ __launch_bounds__(64 * WK, 2) void gemv_awq_wide_kernel(AwqFewParams p) {
  // A wave's 8 KB of each: before the waves meet x of half a chunk, then its sums of rows 0-7 and 8-15.  Two arrays, so that the
  // compiler knows which outstanding load a read has to wait for.
  __shared__ uint4_t ring0[WK * 512];
  __shared__ uint4_t ring1[WK * 512];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kq = lane >> 4;
  const int N = p.N, M = p.M, NC = N >> 3;
  const int tile = blockIdx.x, split = blockIdx.y;
  const int cw = tile * 32 + 2 * j;  // first of the lane's two words
  const int slot = split * WK + wave;
  const int c0 = slot * p.cpw + min(slot, p.rem);
  const int nchunks = p.cpw + (slot < p.rem ? 1 : 0);

  const direct_rsrc_t wrsrc = direct_rsrc(p.qweight, (uint32_t)p.K * (uint32_t)NC * 4u);
  const direct_rsrc_t srsrc = direct_rsrc(p.scales, (uint32_t)p.num_groups * (uint32_t)N * 2u);
  const direct_rsrc_t zrsrc = direct_rsrc(p.qzeros, (uint32_t)p.num_groups * (uint32_t)NC * 4u);
  const direct_rsrc_t xrsrc = direct_rsrc(p.x, (uint32_t)M * (uint32_t)p.K * 2u);
  const uint32_t row_bytes = (uint32_t)NC * 4u;
  const uint32_t w_lane = (uint32_t)(8 * kq) * row_bytes + (uint32_t)cw * 4u;
  // x: load u of half a chunk covers rows 8 u + lane / 8.  A row past M lies past the end of x: no memory is touched, and
  // what the row then holds in LDS only reaches sums that nobody stores.
  uint32_t x_lane[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = 8 * u + (lane >> 3);
    x_lane[u] = ((uint32_t)row * (uint32_t)p.K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 8u) * 2u;
  }

  struct Columns {
    uint4_t s[2];  // sixteen scales
    uint2_t z;
  };
  auto load_x = [&](int c, int h, uint4_t* ring) __attribute__((always_inline)) {
    const uint32_t at = scalar_u32((uint32_t)(c0 + c) * 256u + (uint32_t)h * 128u);
#pragma unroll
    for (int u = 0; u < 2; ++u) load_to_lds(xrsrc, ring + wave * 512 + u * 64, x_lane[u], at);
  };
  auto load_columns = [&](int c, Columns& g) __attribute__((always_inline)) {
    const uint32_t gi = (uint32_t)min((int)(scalar_u32((uint32_t)(c0 + c)) >> p.gshift), p.num_groups - 1);
    g.z = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(zrsrc, (uint32_t)cw * 4u, gi * row_bytes, 0));
    g.s[0] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(srsrc, (uint32_t)cw * 16u, gi * (uint32_t)N * 2u, 0));
    g.s[1] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(srsrc, (uint32_t)cw * 16u, gi * (uint32_t)N * 2u + 16u, 0));
  };
  auto load_step = [&](int c, int st, uint2_t (&w)[8]) __attribute__((always_inline)) {
    const uint32_t at = scalar_u32((uint32_t)(c0 + c) * 128u + (uint32_t)st * 32u) * row_bytes;
#pragma unroll
    for (int r = 0; r < 8; ++r)
      w[r] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(wrsrc, w_lane, at + (uint32_t)r * row_bytes, 2));
    __builtin_amdgcn_sched_barrier(0);
  };

  // fp16 splices for both data types (bf16: the mixed multiply-add reads the halves)
  const LeanConsts kc = lean_consts<Q4_DTYPE_F16>();
  const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  float4_t acc[2][8], part[2][8];  // [word][nibble]
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int f = 0; f < 8; ++f) acc[b][f] = zero4;
  // -(1024 + z) of the even nibbles f, -(64 + z) of the odd ones: component f % 4, half f / 4
  uint32_t cz[2][4];
  auto begin = [&](const Columns& g) __attribute__((always_inline)) {
    const uint32_t zz[2] = {g.z.x, g.z.y};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t z8 = zz[b] >> 8;
      cz[b][0] = (zz[b] & 0x000F000Fu) | 0xE400E400u;
      cz[b][1] = (zz[b] & 0x00F000F0u) | 0xD400D400u;
      cz[b][2] = (z8 & 0x000F000Fu) | 0xE400E400u;
      cz[b][3] = (z8 & 0x00F000F0u) | 0xD400D400u;
    }
  };
  // nibble f of two rows, spliced, minus its constant: exact q - z
  auto minus = [&](uint32_t v, int b, int f) __attribute__((always_inline)) {
    const uint32_t c = cz[b][f & 3];
    if constexpr (DTYPE == Q4_DTYPE_F16) {
      const half2_t h = as_half2(c);
      return as_u32(as_half2(v) + (f < 4 ? half2_t{h.x, h.x} : half2_t{h.y, h.y}));
    } else {
      gemm_float2_t o;
      if (f < 4) {
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,1]" : "=v"(o.x) : "v"(v), "v"(c));
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,1]" : "=v"(o.y) : "v"(v), "v"(c));
      } else {
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[0,0,1] op_sel_hi:[1,0,1]" : "=v"(o.x) : "v"(v), "v"(c));
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(o.y) : "v"(v), "v"(c));
      }
      return __builtin_bit_cast(uint32_t, __builtin_convertvector(o, gemm_bf16x2_t));
    }
  };
  auto process = [&](const uint4_t* ring, int st, const uint2_t (&w)[8]) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const uint4_t a = ring[wave * 512 + j * 8 + (((st & 1) * 4 + kq) ^ ((j >> 1) & 7))];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int by = 0; by < 4; ++by) {
        // byte `by` of two neighbouring rows side by side: nibbles 2 by and 2 by + 1
        const uint32_t sel = 0x0C000C00u | (uint32_t)by | ((uint32_t)(4 + by) << 16);
        uint4_t lo, hi;
#pragma unroll
        for (int rp = 0; rp < 4; ++rp) {
          const uint32_t t = __builtin_amdgcn_perm(b ? w[2 * rp + 1].y : w[2 * rp + 1].x, b ? w[2 * rp].y : w[2 * rp].x, sel);
          lo[rp] = minus((t & kc.mask_lo) | kc.magic_lo, b, 2 * by);
          hi[rp] = minus((t & kc.mask_hi) | kc.magic_hi, b, 2 * by + 1);
        }
        if (st == 0) part[b][2 * by] = part[b][2 * by + 1] = zero4;
        batch_mfma<DTYPE>(a, lo, part[b][2 * by]);
        batch_mfma<DTYPE>(a, hi, part[b][2 * by + 1]);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish_chunk = [&](const uint4_t& s0, const uint4_t& s1) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int f = 0; f < 8; ++f) {
        const uint4_t s = b ? s1 : s0;
        const half2_t sp = as_half2(s[f & 3]);  // nibble f is column 2 (f % 4) + f / 4 of the word
        const float sf = (float)(f < 4 ? sp.x : sp.y);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[b][f][i] = fmaf(sf, part[b][f][i], acc[b][f][i]);
      }
  };

  // Two 32-row steps of weights in flight and the x of one chunk; no load sits behind a branch.
  Columns g;
  uint2_t w[2][8];
  load_x(0, 0, ring0);
  load_columns(0, g);
  load_step(0, 0, w[0]);
  load_x(0, 1, ring1);
  load_step(0, 1, w[1]);
  for (int c = 0; c + 1 < nchunks; ++c) {
    begin(g);
    const uint4_t s0 = g.s[0], s1 = g.s[1];
    load_columns(c + 1, g);
    process(ring0, 0, w[0]);
    load_step(c, 2, w[0]);
    process(ring0, 1, w[1]);
    load_x(c + 1, 0, ring0);
    load_step(c, 3, w[1]);
    process(ring1, 2, w[0]);
    load_step(c + 1, 0, w[0]);
    process(ring1, 3, w[1]);
    load_x(c + 1, 1, ring1);
    load_step(c + 1, 1, w[1]);
    finish_chunk(s0, s1);
  }
  begin(g);
  process(ring0, 0, w[0]);
  load_step(nchunks - 1, 2, w[0]);
  process(ring0, 1, w[1]);
  load_step(nchunks - 1, 3, w[1]);
  process(ring1, 2, w[0]);
  process(ring1, 3, w[1]);
  finish_chunk(g.s[0], g.s[1]);

  // ---- the K waves meet in LDS, each wave's sums where its own x was: lane block kq holds rows 4 kq .. 4 kq + 3, column
  // 16 j + 4 q + i of a row at position 64 q + 4 j + i
  auto sums = [&](int wv, int row) { return (float*)((row & 8) ? ring1 : ring0) + (wv * 8 + (row & 7)) * 256; };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float* const dst = sums(wave, 4 * kq + i);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int b = q >> 1, f = 2 * (q & 1);
      *(float4_t*)(dst + q * 64 + 4 * j) = float4_t{acc[b][f][i], acc[b][f + 4][i], acc[b][f + 1][i], acc[b][f + 5][i]};
    }
  }
  __syncthreads();
  // A unit: 64 lanes with two neighbouring columns each of half a tile row
  constexpr int PP = 2 * kAwqWideRows / WK;
  float v0[PP], v1[PP];
  bool mine[PP];
  auto unit = [&](int e) { return wave + e * WK; };
#pragma unroll
  for (int e = 0; e < PP; ++e) {
    const int row = unit(e) >> 1, at = (unit(e) & 1) * 128 + 2 * lane;
    mine[e] = row < M;
    gemm_float2_t v = *(const gemm_float2_t*)(sums(0, row) + at);
#pragma unroll
    for (int wv = 1; wv < WK; ++wv) v += *(const gemm_float2_t*)(sums(wv, row) + at);
    v0[e] = v.x;
    v1[e] = v.y;
  }

  // ---- workgroups along K meet in pairs, level by level: leaves the sums in a cell, or takes the partner's out of it and goes on
  auto exchange = [&](unsigned long long* plane, size_t row_cells, unsigned long long (&old)[PP]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < PP; ++e) {
      old[e] = 0ull;
      if (mine[e]) {
        // a cell at zero is empty: +0 travels as -0
        uint32_t lo = __builtin_bit_cast(uint32_t, v0[e]);
        lo = lo == 0u ? 0x80000000u : lo;
        const unsigned long long v = (unsigned long long)lo | ((unsigned long long)__builtin_bit_cast(uint32_t, v1[e]) << 32);
        old[e] = __hip_atomic_exchange(plane + unit(e) * row_cells, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
#pragma unroll
    for (int e = 0; e < PP; ++e) {
      mine[e] = old[e] != 0ull;  // the second to arrive carries the sum on
      if (mine[e]) __hip_atomic_store(plane + unit(e) * row_cells, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  const size_t row_cells = (size_t)64 * gridDim.x, plane_cells = (size_t)2 * M * row_cells;
  unsigned long long old[PP];
  int idx = split, meet = 0;
  for (int cnt = p.splits; cnt > 1; cnt = (cnt + 1) >> 1) {
    if ((idx ^ 1) < cnt) {  // (the last of an odd number goes on alone)
      exchange(p.cells + (size_t)(meet + (idx >> 1)) * plane_cells + tile * 64 + lane, row_cells, old);
#pragma unroll
      for (int e = 0; e < PP; ++e)
        if (mine[e]) {
          v0[e] += __builtin_bit_cast(float, (uint32_t)old[e]);
          v1[e] += __builtin_bit_cast(float, (uint32_t)(old[e] >> 32));
        }
    }
    meet += cnt >> 1;
    idx >>= 1;
  }
  const int tiles = FUSE ? (int)gridDim.x >> 1 : (int)gridDim.x;
  const bool up = FUSE && tile >= tiles;
  const int out_tile = up ? tile - tiles : tile;
  // gate tile and up tile meet, behind the cells of all splits
  if constexpr (FUSE) exchange(p.cells + (size_t)(p.splits - 1) * plane_cells + out_tile * 64 + lane, row_cells >> 1, old);

  uint16_t* y = (uint16_t*)p.y;
#pragma unroll
  for (int e = 0; e < PP; ++e) {
    if (!mine[e]) continue;
    const int row = unit(e) >> 1, u = unit(e) & 1;
    const int n = out_tile * 256 + 16 * ((lane >> 1) & 15) + 4 * (2 * u + (lane >> 5)) + 2 * (lane & 1);
    const float a = v0[e] + 0.f, b = v1[e] + 0.f;  // (-0 of an empty sum back to +0)
    uint32_t o0, o1;
    if constexpr (FUSE) {
      const int half = N >> 1;
      const float c = __builtin_bit_cast(float, (uint32_t)old[e]) + 0.f, d = __builtin_bit_cast(float, (uint32_t)(old[e] >> 32)) + 0.f;
      o0 = act_mul<DTYPE>(finish_output<DTYPE>(up ? c : a, p.bias, n), finish_output<DTYPE>(up ? a : c, p.bias, n + half), p.act);
      o1 = act_mul<DTYPE>(finish_output<DTYPE>(up ? d : b, p.bias, n + 1), finish_output<DTYPE>(up ? b : d, p.bias, n + 1 + half), p.act);
      *(uint32_t*)(y + (size_t)row * half + n) = (o0 & 0xFFFFu) | (o1 << 16);
    } else {
      o0 = finish_output<DTYPE>(a, p.bias, n);
      o1 = finish_output<DTYPE>(b, p.bias, n + 1);
      *(uint32_t*)(y + (size_t)row * N + n) = (o0 & 0xFFFFu) | (o1 << 16);
    }
  }
}

}  // namespace q4

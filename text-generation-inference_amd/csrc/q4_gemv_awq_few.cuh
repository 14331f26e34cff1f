// Decode kernel for the AWQ layout (qweight [K, N/8]: a word holds eight interleaved columns of one K row), one to four
// activation rows, optionally with the gated-MLP epilogue.
//
// What bounds it is the stream of packed words, and AWQ's rows make that a matter of the wave tile: 128-column tiles
// read 64-byte pieces of every row, which the memory serves at 60-70 % of the rate of 128-byte ones whatever the
// grid (4096 x 28672, a kernel that only reads: 16.6 us and 10.2; fetching whole lines in two workgroups 17.6).  So a wave owns 256
// columns, two words a lane, and the rest follows from there being few tiles:
//   * The words go into the matrix core as they are stored.  The four K slots that a lane has in a 16x16x16 MFMA are four
//     columns of one K row (half a spliced word; AWQ's interleave yields the columns in order), the A operand is
//     sparse: MFMA row 4 m + c carries x[m][k] in slot c.  One MFMA serves four activation rows and the matrix core
//     adds the four K rows of the lane blocks.  Eleven vector instructions a word; transposing the words into
//     K order costs the batch kernel fourteen and more on this tile.
//   * The splice's offset and the zero point leave a weight before the MFMA, which sums x times the exact integer q - z; the
//     scale multiplies the fp32 sum of a 128-row chunk.  Rows that are not finite need no second look.
//   * No slab and no barrier before the K waves meet: a wave passes the x of its chunk through 1 KB of LDS of its own.
//   * K is dealt in 128-row chunks over K waves and workgroups.  Workgroups along K meet as in the batch kernel (pairs of
//     fp32 sums exchanged), any number of them: an odd one out goes on alone.  (14336 x 4096, one row, 14 workgroups: 10.0 us in
//     four levels, 9.4 with one fixed-point atomic per sum; four rows 11.1 and 11.8.)
//   * Two 32-row steps of a wave are in flight, 8 KB: four measured 3-13 % slower on nine shapes, one 2-25 % (4096 x 28672
//     gated, one row: one step 14.7 us, two 14.4, four 15.2; 4096 x 6144 7.7 / 6.3 / 7.0).
//   * WN = 2: neighbouring tiles, or with the gated epilogue the gate and the up tile, are waves of one workgroup.  As many waves
//     in half as many workgroups fill the CUs evenly where the tiles are many (4096 x 28672, one row: 14.0 us with WN = 1, 13.1).
#pragma once
#include "q4_gemm_kernels.cuh"
#include "q4_gemv_awq.cuh"

namespace q4 {

struct AwqFewParams {
  const uint32_t* __restrict__ qweight;
  const uint32_t* __restrict__ qzeros;
  const half_t* __restrict__ scales;
  const void* __restrict__ x;
  const void* __restrict__ bias;
  void* __restrict__ y;
  unsigned long long* __restrict__ cells;  // exchange cells, zero between launches (splits > 1)
  int N, K, M;
  int cpw, rem;  // 128-row chunks per (split, wave) slot; the first `rem` slots walk one more
  int gshift;    // group of chunk c = min(c >> gshift, num_groups - 1)
  int num_groups;
  int splits;
  int act;
};

constexpr int kAwqFewRows = 4;

// Eight spliced nibbles of a word minus their constants, exact: columns (0,1) (2,3) (4,5) (6,7).
template <int DTYPE>
__device__ __forceinline__ uint4_t awq_few_unpack(uint32_t w, const uint4_t& c, const LeanConsts& k) {
  const uint32_t w8 = w >> 8;
  const uint32_t v[4] = {(w & k.mask_lo) | k.magic_lo, (w & k.mask_hi) | k.magic_hi, (w8 & k.mask_lo) | k.magic_lo, (w8 & k.mask_hi) | k.magic_hi};
  const uint32_t z[4] = {c.x, c.y, c.z, c.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DTYPE == Q4_DTYPE_F16) {
      o[i] = as_u32(as_half2(v[i]) + as_half2(z[i]));
    } else {
      gemm_float2_t f;
      asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,1]" : "=v"(f.x) : "v"(v[i]), "v"(z[i]));
      asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(f.y) : "v"(v[i]), "v"(z[i]));
      o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, gemm_bf16x2_t));
    }
  }
  return uint4_t{o[0], o[1], o[2], o[3]};
}

// WN: column waves (gated epilogue: 2).  WK: K waves.
template <int DTYPE, int WN, int WK, bool FUSE>
__global__ __launch_bounds__(64 * WN * WK, 2) void gemv_awq_few_kernel(AwqFewParams p) {
  static_assert(!FUSE || WN == 2, "gated epilogue: a gate and an up tile");
  constexpr int RING = 2;  // 32-row steps of weights in flight
  constexpr int WAVES = WN * WK;
  __shared__ float sums[WAVES * kAwqFewRows * 256];  // before the waves meet: a wave's first 1 KB holds its x
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kq = lane >> 4;
  const int N = p.N, M = p.M, NC = N >> 3, half = N >> 1;
  const int wn = wave % WN;
  const int tile = blockIdx.x, split = blockIdx.y;
  const int cw = (FUSE ? tile * 32 + wn * (NC >> 1) : (tile * WN + wn) * 32) + 2 * j;  // first of the lane's two words
  const int slot = split * WK + wave / WN;
  const int c0 = slot * p.cpw + min(slot, p.rem);
  const int nchunks = p.cpw + (slot < p.rem ? 1 : 0);

  const direct_rsrc_t wrsrc = direct_rsrc(p.qweight, (uint32_t)p.K * (uint32_t)NC * 4u);
  const direct_rsrc_t srsrc = direct_rsrc(p.scales, (uint32_t)p.num_groups * (uint32_t)N * 2u);
  const direct_rsrc_t zrsrc = direct_rsrc(p.qzeros, (uint32_t)p.num_groups * (uint32_t)NC * 4u);
  const direct_rsrc_t xrsrc = direct_rsrc(p.x, (uint32_t)M * (uint32_t)p.K * 2u);
  const uint32_t row_bytes = (uint32_t)NC * 4u;
  const uint32_t w_lane = (uint32_t)(8 * kq) * row_bytes + (uint32_t)cw * 4u;
  const uint32_t x_lane = ((uint32_t)kq * (uint32_t)p.K + (uint32_t)j * 8u) * 2u;  // (a row past M lies past the end of x: zeros)
  char* const xbuf = (char*)(sums + wave * kAwqFewRows * 256);

  struct Columns {
    uint4_t s[2];  // sixteen scales
    uint2_t z;
  };
  // x, scales and zero points of a chunk, then its first half; the second half.  No load sits behind a branch.
  auto load_head = [&](int c, uint4_t& x, Columns& g) __attribute__((always_inline)) {
    const uint32_t chunk = scalar_u32((uint32_t)(c0 + c));
    const uint32_t gi = (uint32_t)min((int)(chunk >> p.gshift), p.num_groups - 1);
    x = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, x_lane, chunk * 256u, 0));
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
  // A operand: MFMA row j is (activation row j / 4, slot j % 4)
  const uint32_t slot_mask = (j & 1) ? 0xFFFF0000u : 0x0000FFFFu;
  const uint32_t amask0 = (j & 2) ? 0u : slot_mask, amask1 = (j & 2) ? slot_mask : 0u;
  const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  float tot[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) tot[t] = 0.f;
  float4_t acc[2][2];  // [word][half word]
  uint4_t cz[2];       // -(1024 + z), -(64 + z) of the lane's columns
  auto begin = [&](const uint4_t& x, const Columns& g) __attribute__((always_inline)) {
    *(uint4_t*)(xbuf + lane * 16) = x;
    const uint32_t zz[2] = {g.z.x, g.z.y};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t z8 = zz[b] >> 8;
      cz[b] = uint4_t{(zz[b] & 0x000F000Fu) | 0xE400E400u, (zz[b] & 0x00F000F0u) | 0xD400D400u, (z8 & 0x000F000Fu) | 0xE400E400u,
                      (z8 & 0x00F000F0u) | 0xD400D400u};
      acc[b][0] = acc[b][1] = zero4;
    }
  };
  auto process = [&](int st, const uint2_t (&w)[8]) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const uint4_t xa = *(const uint4_t*)(xbuf + (j >> 2) * 256 + st * 64 + kq * 16);
    const uint32_t xp[4] = {xa.x, xa.y, xa.z, xa.w};
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const uint32_t xx = __builtin_amdgcn_perm(xp[r >> 1], xp[r >> 1], (r & 1) ? 0x03020302u : 0x01000100u);
      const uint2_t a = {xx & amask0, xx & amask1};
      const uint4_t u0 = awq_few_unpack<DTYPE>(w[r].x, cz[0], kc), u1 = awq_few_unpack<DTYPE>(w[r].y, cz[1], kc);
      acc[0][0] = diag_mfma<DTYPE>(a, uint2_t{u0.x, u0.y}, acc[0][0]);
      acc[0][1] = diag_mfma<DTYPE>(a, uint2_t{u0.z, u0.w}, acc[0][1]);
      acc[1][0] = diag_mfma<DTYPE>(a, uint2_t{u1.x, u1.y}, acc[1][0]);
      acc[1][1] = diag_mfma<DTYPE>(a, uint2_t{u1.z, u1.w}, acc[1][1]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish_chunk = [&](const uint4_t& s0, const uint4_t& s1) __attribute__((always_inline)) {
    const uint32_t su[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const half2_t sp = as_half2(su[t >> 1]);
      tot[t] = fmaf((float)((t & 1) ? sp.y : sp.x), acc[t >> 3][(t >> 2) & 1][t & 3], tot[t]);
    }
  };

  uint4_t x;
  Columns g;
  uint2_t w[RING][8];
  load_head(0, x, g);
#pragma unroll
  for (int st = 0; st < RING; ++st) load_step(0, st, w[st]);
  for (int c = 0; c + 1 < nchunks; ++c) {
    begin(x, g);
    const uint4_t s0 = g.s[0], s1 = g.s[1];
    load_head(c + 1, x, g);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      process(st, w[st % RING]);
      load_step(c + (st + RING) / 4, (st + RING) % 4, w[st % RING]);
    }
    finish_chunk(s0, s1);
  }
  begin(x, g);
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    process(st, w[st % RING]);
    if (st + RING < 4) load_step(nchunks - 1, st + RING, w[st % RING]);
  }
  finish_chunk(g.s[0], g.s[1]);

  // ---- the K waves meet in LDS: lane block kq holds row kq, its 16 columns four at a time so that neighbouring lanes write
  // neighbouring 16 bytes (position 64 q + 4 j + i of a row is column 16 j + 4 q + i)
  if (kq < M) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(float4_t*)(sums + (wave * kAwqFewRows + kq) * 256 + q * 64 + 4 * j) = float4_t{tot[4 * q], tot[4 * q + 1], tot[4 * q + 2], tot[4 * q + 3]};
  }
  __syncthreads();
  // A unit: 64 lanes with two sums each, neighbouring columns of half a tile row, or the gate and up sums of a quarter
  constexpr int UNITS = FUSE ? 4 : 2 * WN;  // of a row
  constexpr int PP = UNITS * kAwqFewRows / WAVES;
  static_assert(PP * WAVES == UNITS * kAwqFewRows, "units are dealt evenly");
  float v0[PP], v1[PP];
  bool mine[PP];
  auto unit = [&](int e) { return wave + e * WAVES; };
  auto sum_at = [&](int wn0, int row, int pos, auto& v) {
    v = 0;
#pragma unroll
    for (int w = 0; w < WK; ++w) v += *(const std::remove_reference_t<decltype(v)>*)(sums + ((w * WN + wn0) * kAwqFewRows + row) * 256 + pos);
  };
#pragma unroll
  for (int e = 0; e < PP; ++e) {
    const int row = unit(e) / UNITS, u = unit(e) % UNITS;
    mine[e] = row < M;
    v0[e] = v1[e] = 0.f;
    if (mine[e]) {
      if constexpr (FUSE) {
        sum_at(0, row, u * 64 + lane, v0[e]);
        sum_at(1, row, u * 64 + lane, v1[e]);
      } else {
        gemm_float2_t v;
        sum_at(u >> 1, row, (u & 1) * 128 + 2 * lane, v);
        v0[e] = v.x;
        v1[e] = v.y;
      }
    }
  }

  // ---- workgroups along K meet in pairs, level by level: leaves the sums in a cell, or takes the partner's out of it and goes on
  const size_t row_cells = (size_t)64 * gridDim.x, plane_cells = (size_t)UNITS * M * row_cells;
  int idx = split, meet = 0;
  for (int cnt = p.splits; cnt > 1; cnt = (cnt + 1) >> 1) {
    if ((idx ^ 1) < cnt) {  // (the last of an odd number goes on alone)
      unsigned long long* plane = p.cells + (size_t)(meet + (idx >> 1)) * plane_cells + tile * 64 + lane;
      unsigned long long old[PP];
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
        if (mine[e]) {
          __hip_atomic_store(plane + unit(e) * row_cells, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          v0[e] += __builtin_bit_cast(float, (uint32_t)old[e]);
          v1[e] += __builtin_bit_cast(float, (uint32_t)(old[e] >> 32));
        }
      }
    }
    meet += cnt >> 1;
    idx >>= 1;
  }

  uint16_t* y = (uint16_t*)p.y;
#pragma unroll
  for (int e = 0; e < PP; ++e) {
    if (!mine[e]) continue;
    const int row = unit(e) / UNITS, u = unit(e) % UNITS;
    const float a = v0[e] + 0.f, b = v1[e] + 0.f;  // (-0 of an empty sum back to +0)
    if constexpr (FUSE) {
      const int n = tile * 256 + 16 * (lane >> 2) + 4 * u + (lane & 3);
      y[(size_t)row * half + n] = act_mul<DTYPE>(finish_output<DTYPE>(a, p.bias, n), finish_output<DTYPE>(b, p.bias, n + half), p.act);
    } else {
      const int n = (tile * WN + (u >> 1)) * 256 + 16 * ((lane >> 1) & 15) + 4 * (2 * (u & 1) + (lane >> 5)) + 2 * (lane & 1);
      *(uint32_t*)(y + (size_t)row * N + n) = finish_output<DTYPE>(a, p.bias, n) | ((uint32_t)finish_output<DTYPE>(b, p.bias, n + 1) << 16);
    }
  }
}

}  // namespace q4

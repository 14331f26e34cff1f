// Prefill kernel with one wave per SIMD: y[M, N] = x @ dequant(W), GPTQ layout with contiguous groups and AWQ layout,
// optionally with the gated-MLP epilogue.
//
// What bounds prefill is the matrix pipes, and with every CU at work the power they may draw: padded rows and
// repeated unpacking cost as much as useful work.  So the height of the tile follows M (32 R rows x 256 columns, R = 3 ..
// 6 or 8) and every weight is unpacked once per tile:
//   * Four waves side by side along N, 64 columns each, all 32 R rows: 32 R accumulators of a 512-register budget.
//     Nothing else runs on a SIMD, so a wave overlaps by itself: the words of the next 16-row step are
//     unpacked between this step's v_mfma_f32_32x32x16 (eight passes each; the vector instructions find room in
//     their shadow.  Between 16x16x32 ones, which keep the register ports busy, they do not: 160 rows, K tile of 64 rows,
//     0.83 us against 1.0).
//   * The activation tile (32 R rows x 64 K) goes from memory straight into LDS (buffer_load ... lds), a ring of four
//     tiles, asked for three ahead; 16-byte units XOR swizzled by row on the global side (7-11 % of the LDS
//     cycles go to bank conflicts, 256 x 256 tiles 8 %; waves wait at most 1 % of their time for LDS); one barrier per K tile.
//   * The activations stay in their own K order, so GPTQ words are unpacked byte by byte (16 operations per word of eight).
// Measured on MI355X, us, 128 x 256 tiles (two workgroups per CU, 384 rows padded) / this kernel with 160-row
// tiles: 4096 x 28672 gated at 301 rows 109 / 78, 14336 x 4096 57 / 49.
// GPTQ tiles of up to 160 rows may split K inside the workgroup (KW = 2): two column waves times two halves of K, each half with its own ring of
// activation tiles (160 KB of LDS at 160 rows), whose sums meet in LDS.  Half the partial sums that go through memory for as many
// workgroups: 3584 x 8192 at 301 rows 34.4 us / 28.9; the rule is tall_plan's.
// Quantisation groups are multiples of 64 rows (one group per K tile).
#pragma once

#include "q4_gemm_awq_direct.cuh"

namespace q4 {

constexpr int kTallBN = 256;
constexpr int kTileGptq = 0, kTileAwq = 1;

// Constants of one GPTQ column within one quantisation group, for weights in natural K order.
template <int DTYPE>
struct WordCol;
template <>
struct WordCol<Q4_DTYPE_F16> {
  half2_t cz;  // (-(1024 + z), -(64 + z))
  half2_t s2;  // (s, s)
};
template <>
struct WordCol<Q4_DTYPE_BF16> {
  float sf, clo, chi;  // float(s), -(1024 + z) * float(s), -(64 + z) * float(s): exact
};
template <int DTYPE>
__device__ __forceinline__ WordCol<DTYPE> make_word_col(uint32_t z, half_t s) {
  WordCol<DTYPE> c;
  if constexpr (DTYPE == Q4_DTYPE_F16) {
    c.cz = as_half2(0xD400E400u | z | (z << 20));
    c.s2 = half2_t{s, s};
  } else {
    c.sf = (float)s;
    c.clo = -(1024.f + (float)z) * c.sf;
    c.chi = -(64.f + (float)z) * c.sf;
  }
  return c;
}

struct WordK {
  uint32_t mask, magic;
};
__device__ __forceinline__ WordK word_consts() {
  WordK k{0x00F0000Fu, 0x54006400u};  // register operands, so that (t & mask) | magic selects v_and_or_b32
  asm volatile("" : "+s"(k.mask), "+v"(k.magic));
  return k;
}

// Byte b of a packed GPTQ word -> weights 2 b and 2 b + 1 of one column.  The byte in both halves of a register: its low
// nibble spliced into 1024 (1024 + q) below, its high nibble into 64 (mantissa step 1/16: 64 + q) above.
template <int DTYPE>
__device__ __forceinline__ uint32_t dequant_byte(uint32_t w, int b, const WordCol<DTYPE>& c, const WordK& k) {
  const uint32_t v = (__builtin_amdgcn_perm(w, w, 0x0C000C00u | (uint32_t)b | ((uint32_t)b << 16)) & k.mask) | k.magic;
  if constexpr (DTYPE == Q4_DTYPE_F16) {
    return as_u32((as_half2(v) + c.cz) * c.s2);  // exact q - z, then the reference's one fp16 rounding
  } else {
    gemm_float2_t f;  // exact in fp32, rounded once by the packed convert
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(f.x) : "v"(v), "v"(c.sf), "v"(c.clo));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(f.y) : "v"(v), "v"(c.sf), "v"(c.chi));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, gemm_bf16x2_t));
  }
}

// Half of awq_unpack_pair: the two fragments of one byte of two consecutive rows' words.
template <int DTYPE>
__device__ __forceinline__ void awq_unpack_half(uint32_t w0, uint32_t w1, uint32_t sel, const AwqCol<DTYPE>& cl,
                                                const AwqCol<DTYPE>& ch, const AwqSpliceK& k, uint32_t& lo, uint32_t& hi) {
  const uint32_t t = __builtin_amdgcn_perm(w1, w0, sel);
  const uint32_t v[2] = {(t & k.mask_lo) | k.magic_lo, (t & k.mask_hi) | k.magic_hi};
  uint32_t o[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const AwqCol<DTYPE>& c = f == 0 ? cl : ch;
    if constexpr (DTYPE == Q4_DTYPE_F16) {
      o[f] = as_u32((as_half2(v[f]) + c.cz) * c.s2);
    } else {
      gemm_float2_t t2;
      asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(t2.x) : "v"(v[f]), "v"(c.sf), "v"(c.cf));
      asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(t2.y) : "v"(v[f]), "v"(c.sf), "v"(c.cf));
      o[f] = __builtin_bit_cast(uint32_t, __builtin_convertvector(t2, gemm_bf16x2_t));
    }
  }
  lo = o[0];
  hi = o[1];
}

// KW = 2: the workgroup's waves are two column waves times two halves of its K range, which meet in LDS; its tile is 128 columns.
template <int DTYPE, int LAYOUT, int R, bool FUSE, int KW = 1>
__global__ __launch_bounds__(256, 1) void gemm_tall_kernel(GemmParams gp) {
  static_assert(KW == 1 || (!FUSE && R <= 5), "two K halves: plain launches, whose rings fit LDS");
  constexpr bool AWQ = LAYOUT == kTileAwq;
  constexpr int BM = 32 * R;
  constexpr int WAVES = 4;
  constexpr int A_BLOCKS = BM / 8;                // 8 rows x 128 bytes of the activation tile: one load of a wave
  constexpr int CW = WAVES / KW;                       // column waves, which load their K half's tile
  constexpr int BN = kTallBN / KW;
  constexpr int A_LOADS = A_BLOCKS / CW;               // of a wave
  constexpr int FR = kKSteps * R;                  // A fragments of a wave per K tile
  // four arrays: the compiler then knows which outstanding load a fragment read has to wait for
  __shared__ uint4_t ring0[KW * BM * 8], ring1[KW * BM * 8], ring2[KW * BM * 8], ring3[KW * BM * 8];
  const Problem& p = gp.p;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (WAVES - 1);  // (known range: LDS addresses fold into offsets)
  const int cw = wave % CW, kh = wave / CW;  // column wave, K half
  const int j = lane & 31;
  const int kq = lane >> 5;
  const int N = p.N, K = p.K, M = p.M;

  // Tile order: workgroup ids go round-robin over the 8 XCDs.  More than one round: every XCD keeps its own
  // M tiles (activations in its L2) and walks the column blocks; otherwise it takes a few column blocks and
  // all their M tiles.
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = N / BN;
  const int total = tiles_m * tiles_n;
  const int split = blockIdx.x / total;
  int tm, tn;
  {
    const int bid = blockIdx.x - split * total;
    if (tiles_m % 8 == 0 && total > 256) {
      const int mpx = tiles_m >> 3, local = bid >> 3;
      tm = (bid & 7) * mpx + local % mpx;
      tn = local / mpx;
    } else if (total % 8 == 0) {
      const int lin = (bid & 7) * (total >> 3) + (bid >> 3);
      tm = lin % tiles_m;
      tn = lin / tiles_m;
    } else {
      tm = bid % tiles_m;
      tn = bid / tiles_m;
    }
  }
  const int m0 = tm * BM;
  const int half = N >> 1;
  // first column of this wave (gated epilogue: waves wave = 0, 1 the gate columns, 2, 3 the up columns that go with them)
  const int nw = FUSE ? tn * (kTallBN / 2) + (wave & 1) * 64 + (wave >> 1) * half : tn * BN + cw * 64;
  // the two columns this lane finishes start here; AWQ: lane j unpacks byte j % 4 of word j / 4, columns acol and acol + 2
  const int ncol = AWQ ? nw + 8 * (j >> 2) + ((j & 1) << 2) + (j & 2) : nw + 2 * j;
  const int acol = nw + 8 * (j >> 2) + ((j & 1) << 2) + ((j >> 1) & 1);

  const int KT_all = K / kBK;
  // (KW = 2: the host sees to whole halves)
  const int kt_first = (int)((long)split * KT_all / gp.splits), kt_count = (int)((long)(split + 1) * KT_all / gp.splits) - kt_first;
  const int KT = kt_count / KW, kt0 = kt_first + kh * KT;
  const int last_tile = KT - 1;

  // ---- packed words of a 16-row step.  GPTQ: row 8 kt + 2 s + kq, columns ncol, ncol + 1.  AWQ: rows
  // 64 kt + 16 s + 8 kq + r, r = 0 .. 7, word j / 4 of the wave's eight.
  constexpr int WORDS = AWQ ? 8 : 2;
  constexpr int BSETS = AWQ ? 1 : 2;  // K tiles in flight
  const buffer_rsrc_t wrsrc = make_rsrc(p.qweight, (uint32_t)(K >> 3) * (uint32_t)N * 4u);  // host: below 4 GB
  const uint32_t row_bytes = (uint32_t)N >> 1;  // AWQ: one K row
  const uint32_t w_lane = AWQ ? (uint32_t)(kq * 8) * row_bytes + (uint32_t)((nw >> 3) + (j >> 2)) * 4u
                              : ((uint32_t)kq * (uint32_t)N + (uint32_t)ncol) * 4u;
  const uint32_t step_bytes = (uint32_t)N * 8u;  // 16 K rows
  struct BWords { uint32_t v[WORDS]; };
  BWords bq[BSETS][kKSteps];
  auto load_b = [&](int kt, int s, BWords& dst) {
    const uint32_t off = uniform_u32((uint32_t)((kt0 + kt) * kKSteps + s) * step_bytes);
    if constexpr (AWQ) {
#pragma unroll
      for (int r = 0; r < 8; ++r)
        dst.v[r] = __builtin_amdgcn_raw_buffer_load_b32(wrsrc, w_lane, uniform_u32(off + (uint32_t)r * row_bytes), 0);
    } else {
      const uint2_t t = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(wrsrc, w_lane, off, 0));
      dst.v[0] = t.x; dst.v[1] = t.y;
    }
  };

  // ---- group constants of the lane's two columns, rebuilt for every tile from small loads two tiles ahead
  const buffer_rsrc_t srsrc = make_rsrc(p.scales, (uint32_t)p.num_groups * (uint32_t)N * 2u);
  const buffer_rsrc_t zrsrc = make_rsrc(p.qzeros, (uint32_t)p.num_groups * (uint32_t)(N >> 3) * 4u);
  struct GroupRaw { uint32_t s0, s1, z; };
  GroupRaw raw[2];
  auto load_group_raw = [&](int kt, GroupRaw& g) {
    int gi = ((kt0 + kt) * kBK) / p.groupsize;
    gi = min(gi, p.num_groups - 1);
    const uint32_t srow = uniform_u32((uint32_t)gi * (uint32_t)N * 2u), zrow = uniform_u32((uint32_t)gi * (uint32_t)(N >> 3) * 4u);
    if constexpr (AWQ) {
      g.s0 = __builtin_amdgcn_raw_buffer_load_b16(srsrc, (uint32_t)acol * 2u, srow, 0);
      g.s1 = __builtin_amdgcn_raw_buffer_load_b16(srsrc, (uint32_t)acol * 2u + 4u, srow, 0);
    } else {
      g.s0 = __builtin_amdgcn_raw_buffer_load_b32(srsrc, (uint32_t)ncol * 2u, srow, 0);
    }
    g.z = __builtin_amdgcn_raw_buffer_load_b32(zrsrc, (uint32_t)(ncol >> 3) * 4u, zrow, 0);
  };
  const WordK word_k = word_consts();
  const AwqSpliceK awq_splice = awq_splice_consts();
  const uint32_t sel = 0x0C040C00u + (uint32_t)(j & 3) * 0x00010001u;  // AWQ: byte j % 4 of the words of a row pair
  WordCol<DTYPE> cc[2];
  AwqCol<DTYPE> ac[2];
  auto make_group = [&](const GroupRaw& g) {
    if constexpr (AWQ) {
      const uint32_t z2 = g.z >> (8 * (j & 3));
      ac[0] = make_awq_col<DTYPE, false>(z2 & 0xFu, g.s0);
      ac[1] = make_awq_col<DTYPE, true>((z2 >> 4) & 0xFu, g.s1);
    } else {
      const uint32_t z2 = gptq_zero_plus_one(g.z) >> ((ncol & 7) * 4);
      const half2_t s01 = as_half2(g.s0);
      cc[0] = make_word_col<DTYPE>(z2 & 0xFu, s01.x);
      cc[1] = make_word_col<DTYPE>((z2 >> 4) & 0xFu, s01.y);
    }
  };

  // ---- activation tile: global -> LDS.  Load i of a wave covers rows 8 (cw + CW i) .. + 7, the LDS unit lane % 8 of a
  // row receives its unit (lane % 8) ^ (row / 2 % 8).
  const buffer_rsrc_t xrsrc = make_rsrc(p.x, (uint32_t)M * (uint32_t)K * 2u);  // host: below 2 GB
  // Rows past M lie past the end of x: such a load touches no memory.
  const int a_row0 = 8 * cw + (lane >> 3);
  const uint32_t a_off0 = ((uint32_t)(m0 + a_row0) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((a_row0 >> 1) & 7)) * 8u) * 2u;
  const uint32_t a_step = (uint32_t)K * (16u * CW);  // 8 CW rows
  auto load_a = [&](int kt, uint4_t* ring) {
    const uint32_t tile_off = uniform_u32((uint32_t)(kt0 + min(kt, last_tile)) * (kBK * 2));
    uint32_t off = a_off0;
    asm volatile("" : "+v"(off));  // (added up for every tile: as loop invariants the sums cost a register each)
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) load_to_lds(xrsrc, ring + kh * (BM * 8) + (cw + CW * i) * 64, off + (uint32_t)i * a_step, tile_off);
  };

  float16_t acc[R][2];
#pragma unroll
  for (int mt = 0; mt < R; ++mt)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][f][r] = 0.f;

  // A fragment g of a tile (g = s * R + mt): the wave's rows 32 mt + j, K unit 2 s + kq (swizzled)
  const int a_swz = (j >> 1) & 7;
  const int a_row = kh * (BM * 8) + j * 8;
  int a_lane[kKSteps];
#pragma unroll
  for (int s = 0; s < kKSteps; ++s) a_lane[s] = a_row + ((2 * s + kq) ^ a_swz);
  constexpr int AHEAD = 2;  // fragments read ahead
  constexpr int SLOTS = AHEAD + 2;
  uint4_t afrag[SLOTS];  // rolling window: fragment g sits in slot g % SLOTS
  auto read_a = [&](const uint4_t* ring, int g) { return ring[a_lane[g / R] + (g % R) * 32 * 8]; };
  uint4_t bfrag[2][2];  // this step's fragments and the next one's

  // unit u of a step's unpacking.  GPTQ: byte u % 4 of word u / 4; AWQ: the lane's byte of two rows' words
  constexpr int UNITS = AWQ ? 4 : 8;
  auto unpack = [&](const BWords& w, int u, uint4_t (&dst)[2]) {
    if constexpr (AWQ) {
      uint32_t lo, hi;
      awq_unpack_half<DTYPE>(w.v[2 * u], w.v[2 * u + 1], sel, ac[0], ac[1], awq_splice, lo, hi);
      dst[0][u] = lo;
      dst[1][u] = hi;
    } else {
      dst[u >> 2][u & 3] = dequant_byte<DTYPE>(w.v[u >> 2], u & 3, cc[u >> 2], word_k);
    }
  };

  load_a(0, ring0);
  load_a(1, ring1);
  load_a(2, ring2);
#pragma unroll
  for (int b = 0; b < BSETS; ++b)
#pragma unroll
    for (int s = 0; s < kKSteps; ++s) load_b(min(b, last_tile), s, bq[b][s]);
  load_group_raw(0, raw[0]);
  load_group_raw(min(1, last_tile), raw[1]);
  make_group(raw[0]);
  load_group_raw(min(2, last_tile), raw[0]);
#pragma unroll
  for (int u = 0; u < UNITS; ++u) unpack(bq[0][0], u, bfrag[0]);
  load_b(min(BSETS, last_tile), 0, bq[0][0]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first tiles are in LDS
  __syncthreads();

  // One K tile: the activation tile three ahead is asked for, then four steps of 2 R MFMAs, each with the A fragments
  // read two ahead, the next step's words unpacked in between and their registers refilled BSETS tiles on.  Tile
  // indices past the end are clamped (fetched again, ignored): no branches.
  auto tile_step = [&](int kt, auto par_c, uint4_t* cur, uint4_t* nxt, uint4_t* free) {
    constexpr int par = decltype(par_c)::value % BSETS, npar = (decltype(par_c)::value + 1) % BSETS;
    constexpr int gn = (decltype(par_c)::value + 1) % 2;
    uint32_t arrived;
    load_a(kt + 3, free);
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) afrag[g] = read_a(cur, g);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kKSteps; ++s) {
      constexpr int LAST = kKSteps - 1;
      BWords& words = s < LAST ? bq[par][s + 1 < kKSteps ? s + 1 : 0] : bq[npar][0];
      if (s == LAST) {
        make_group(raw[gn]);  // the next tile's group
        load_group_raw(min(kt + 3, last_tile), raw[gn]);
      }
#pragma unroll
      for (int mt = 0; mt < R; ++mt) {
        const int g = s * R + mt;
        if (g + AHEAD < FR) afrag[(g + AHEAD) % SLOTS] = read_a(cur, g + AHEAD);
        // a read of the next tile's array: the compiler waits for this wave's loads into it, and for no later ones
        if (g == FR - 2) arrived = nxt[a_lane[0]].x;
#pragma unroll
        for (int u = mt * UNITS / R; u < (mt + 1) * UNITS / R; ++u) unpack(words, u, bfrag[(s + 1) & 1]);
#pragma unroll
        for (int f = 0; f < 2; ++f) acc[mt][f] = mfma32<DTYPE>(afrag[g % SLOTS], bfrag[s & 1][f], acc[mt][f]);
        // an LDS read, then vector instructions under every MFMA
        __builtin_amdgcn_sched_group_barrier(0x080, 1, 0);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      load_b(s < LAST ? min(kt + BSETS, last_tile) : min(kt + 1 + BSETS, last_tile), (s + 1) & LAST, words);
    }
    // Behind the barrier every wave's share of the next tile has arrived and every wave is done with this tile.
    asm volatile("" ::"v"(arrived) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  {
    int kt = 0;
    for (; kt + 3 < KT; kt += 4) {
      tile_step(kt, I0{}, ring0, ring1, ring3);
      tile_step(kt + 1, I1{}, ring1, ring2, ring0);
      tile_step(kt + 2, std::integral_constant<int, 2>{}, ring2, ring3, ring1);
      tile_step(kt + 3, std::integral_constant<int, 3>{}, ring3, ring0, ring2);
    }
    if (kt < KT) tile_step(kt, I0{}, ring0, ring1, ring3);
    if (kt + 1 < KT) tile_step(kt + 1, I1{}, ring1, ring2, ring0);
    if (kt + 2 < KT) tile_step(kt + 2, std::integral_constant<int, 2>{}, ring2, ring3, ring1);
  }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the tiles asked for past the end still write the ring)

  if constexpr (KW == 2) {
    // The K halves hand each other half of their sums through LDS (a column wave's in one array, 8 R KB): half 0 finishes registers 0 .. 7 of
    // every fragment, half 1 the others.
    __syncthreads();
    float4_t* xch = (float4_t*)(cw ? ring1 : ring0) + lane;
#pragma unroll
    for (int mt = 0; mt < R; ++mt)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float4_t v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = kh ? acc[mt][f][4 * q + i] : acc[mt][f][8 + 4 * q + i];
          xch[(((kh * R + mt) * 2 + f) * 2 + q) * 64] = v;
        }
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < R; ++mt)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const float4_t v = xch[((((1 - kh) * R + mt) * 2 + f) * 2 + q) * 64];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mt][f][4 * q + i] = (kh ? acc[mt][f][8 + 4 * q + i] : acc[mt][f][4 * q + i]) + v[i];
        }
  }
  constexpr int REGS = 16 / KW;  // of a fragment that the wave finishes, from 8 kh on

  // ---- epilogue.  C layout of the 32x32 MFMA: register r of lane (j, kq) is row 8 (r / 4) + 4 kq + r % 4, column j of
  // the fragment.  GPTQ: fragment f is column ncol + f.  AWQ: columns acol, acol + 2; lanes j and j ^ 2 swap one of
  // their two sums, then each owns ncol and ncol + 1 as well.
  auto sums = [&](int mt, int r) {
    const float a = acc[mt][0][r], b = acc[mt][1][r];
    if constexpr (AWQ) {
      const bool hi = (j & 2) != 0;
      const float got = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, hi ? a : b), 0x4E, 0xF, 0xF, true));
      return hi ? float2_t{got, b} : float2_t{a, got};
    } else {
      return float2_t{a, b};
    }
  };
  auto row_of = [&](int mt, int r) { return m0 + mt * 32 + (KW == 2 ? 16 * kh : 0) + 8 * (r >> 2) + 4 * kq + (r & 3); };
  if (gp.splits > 1) {
    // fp32 partial tile; bias, rounding and the store to y happen in the reduction kernel
    float* part = gp.partials + (size_t)split * gp.partial_rows * N;
#pragma unroll
    for (int mt = 0; mt < R; ++mt)
#pragma unroll
      for (int r = 0; r < REGS; ++r) {
        const int m = row_of(mt, r);
        const float2_t v = sums(mt, r);
        if (m < M) *(float2_t*)(part + (size_t)m * N + ncol) = v;
      }
    return;
  }
  uint16_t* y = (uint16_t*)p.y;
  const bool has_bias = p.bias != nullptr;
  float bias_f[2] = {0.f, 0.f};
  if (has_bias) {
    bias_f[0] = load_act<DTYPE>(p.bias, ncol);
    bias_f[1] = load_act<DTYPE>(p.bias, ncol + 1);
  }
  // the sum is rounded to the activation dtype first and the bias added in that dtype
  auto finish = [&](float v, float b) -> uint32_t {
    uint16_t o = store_act<DTYPE>(v);
    if (has_bias) {
      float ob;
      if constexpr (DTYPE == Q4_DTYPE_F16) ob = (float)__builtin_bit_cast(half_t, o);
      else ob = bf16_bits_to_f32(o);
      o = store_act<DTYPE>(ob + b);
    }
    return o;
  };
  auto finish2 = [&](int mt, int r) {
    const float2_t v = sums(mt, r);
    return finish(v.x, bias_f[0]) | (finish(v.y, bias_f[1]) << 16);
  };
  if constexpr (FUSE) {
    // act(gate) * up on the rounded halves (what the two-kernel route computes).  The gate and the up wave of
    // a column block hand each other half of their registers through LDS (the activation tiles are dead) and
    // finish the other half: the gate wave registers 0 .. 7 of every block, the up wave 8 .. 15.
    const bool up = wave >= 2;
    __syncthreads();  // (everybody's)
    uint32_t* xch = (uint32_t*)(wave & 1 ? ring1 : ring0) + lane;  // (one pair of waves per array: all of its R x 4 KB)
    uint32_t own[R][8];  // the rounded halves this wave finishes
#pragma unroll
    for (int mt = 0; mt < R; ++mt)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const uint32_t lo = finish2(mt, r), hi = finish2(mt, r + 8);
        own[mt][r] = up ? hi : lo;
        xch[((up ? 0 : R) + mt) * 512 + r * 64] = up ? lo : hi;
      }
    __syncthreads();
    const int oc = up ? ncol - half : ncol;
    auto products = [&](auto act_c) {
      constexpr int ACT = decltype(act_c)::value;
#pragma unroll
      for (int mt = 0; mt < R; ++mt)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const uint32_t other = xch[((up ? R : 0) + mt) * 512 + r * 64];
          const uint32_t g = up ? other : own[mt][r], u = up ? own[mt][r] : other;
          const uint32_t o = (uint32_t)act_mul_as<DTYPE, ACT>((uint16_t)(g & 0xFFFFu), (uint16_t)(u & 0xFFFFu)) |
                             ((uint32_t)act_mul_as<DTYPE, ACT>((uint16_t)(g >> 16), (uint16_t)(u >> 16)) << 16);
          const int m = row_of(mt, r) + (up ? 16 : 0);
          if (m < M) *(uint32_t*)(y + (size_t)m * half + oc) = o;
        }
    };
    const int act = p.gate_up_act - 1;
    if (act == Q4_ACT_SILU) products(std::integral_constant<int, Q4_ACT_SILU>{});
    else if (act == Q4_ACT_GELU_TANH) products(std::integral_constant<int, Q4_ACT_GELU_TANH>{});
    else products(std::integral_constant<int, Q4_ACT_GELU>{});
    return;
  }
#pragma unroll
  for (int mt = 0; mt < R; ++mt)
#pragma unroll
    for (int r = 0; r < REGS; ++r) {
      const int m = row_of(mt, r);
      const uint32_t o = finish2(mt, r);
      if (m < M) *(uint32_t*)(y + (size_t)m * N + ncol) = o;
    }
}

}  // namespace q4

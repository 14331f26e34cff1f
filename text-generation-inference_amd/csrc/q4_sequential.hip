// Act-order without per-weight lookups: the rows of a GPTQ matrix are put into group order
// once at load time and the activation columns follow the same order at run time, after which
// the contiguous-group kernels apply.  The reference's exllamav2 path does the same
// (QMatrix::make_sequential + make_sequential_kernel, cuda/q_matrix.cu:524-640, and the
// b_q_perm gather of the activations in its GEMM, cuda/q_gemm_kernel_gptq.cuh:116).
#include "q4_common.cuh"

namespace q4 {

// out word (r, n) = nibbles of source rows perm[8r .. 8r+7] of column n.  One thread per
// column and packed row: the eight source words are coalesced along n.
__global__ __launch_bounds__(256) void make_sequential_kernel(const uint32_t* __restrict__ qweight,
                                                              const int32_t* __restrict__ perm,
                                                              uint32_t* __restrict__ out, int K, int N) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int r = blockIdx.y;
  if (n >= N) return;
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int src = min(max(perm[8 * r + i], 0), K - 1);  // a bad index reads a wrong row, never outside
    const uint32_t w = qweight[(size_t)(src >> 3) * N + n];
    word |= ((w >> ((src & 7) * 4)) & 0xFu) << (4 * i);
  }
  out[(size_t)r * N + n] = word;
}

// The row order by group, found inside a forward call (q4_linear_regroup) from g_idx as it is in memory then.
// Workgroup g scans all of g_idx (K entries from L2) and writes the rows of group g, ascending, to perm[g
// groupsize ..]; uneven[g] says whether they were not exactly `groupsize`.  perm is valid whatever g_idx holds:
// rows beyond a group's share are left out, missing ones become 0.
__global__ __launch_bounds__(512) void group_order_kernel(const int32_t* __restrict__ g_idx, int32_t* __restrict__ perm,
                                                          int32_t* __restrict__ uneven, int K, int groupsize) {
  __shared__ int sums[8];
  const int g = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int per = ((K >> 2) + 511) / 512 * 4;  // entries of a thread, contiguous
  const int k0 = min(tid * per, K), k1 = min(k0 + per, K);
  int count = 0;
#pragma unroll 4
  for (int k = k0; k < k1; k += 4) {
    const uint4_t v = *(const uint4_t*)(g_idx + k);
    count += ((int)v.x == g) + ((int)v.y == g) + ((int)v.z == g) + ((int)v.w == g);
  }
  int scan = count;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int below = __shfl_up(scan, d);
    if (lane >= d) scan += below;
  }
  if (lane == 63) sums[tid >> 6] = scan;
  __syncthreads();
  int rank = scan - count, total = 0;
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    if (w < (tid >> 6)) rank += sums[w];
    total += sums[w];
  }
  int32_t* dst = perm + (size_t)g * groupsize;
  for (int k = k0; count > 0 && k < k1; k += 4) {
    const uint4_t v = *(const uint4_t*)(g_idx + k);
    const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if ((int)e[i] != g) continue;
      if (rank < groupsize) dst[rank] = k + i;
      ++rank;
    }
  }
  for (int r = total + tid; r < groupsize; r += 512) dst[r] = 0;
  if (tid == 0) uneven[g] = total != groupsize ? 1 : 0;
}

// The same for a whole matrix inside a forward call (q4_linear_regroup).  A source word's nibbles go to
// eight different output words: one thread per word in output order reads everything eight times
// (8192 x 10240: 33 us whether the last-level cache or the L2 serves it, 2.5 TB/s in and out).  Here a
// workgroup holds a panel of C columns over all of K in LDS (K C / 2 bytes: 32 columns up to K = 9600, 16
// or 8 beyond), so memory sees every word once in and once out, and gathers from there: a lane owns four
// adjacent columns of an output row, eight 128-bit LDS reads and two operations per nibble.
// Workgroup 0 also gathers what group_order_kernel found: *any_uneven is 1 if a group has not its share of rows.
template <int C>
__global__ __launch_bounds__(1024) void regroup_kernel(const uint32_t* __restrict__ qweight, const int32_t* __restrict__ perm,
                                                       const int32_t* __restrict__ uneven, int num_groups,
                                                       int32_t* __restrict__ any_uneven, uint32_t* __restrict__ out, int K,
                                                       int N) {
  extern __shared__ __align__(16) uint4_t panel[];  // [K / 8][C / 4]
  constexpr int UPR = C / 4;  // 16-byte units per row
  const int rows = K >> 3, units = rows * UPR;
  if (blockIdx.x == 0) {
    int bad = 0;
    for (int g = threadIdx.x; g < num_groups; g += 1024) bad |= uneven[g];
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) *any_uneven = bad != 0 ? 1 : 0;
  }
  // Panels narrower than a cache line: the ones that share lines run on one XCD (workgroup ids go to the 8
  // XCDs in turn), whose L2 then fetches a line once and collects its parts on the way out.
  constexpr int SHARE = 32 / C;
  int p = blockIdx.x;
  if (SHARE > 1 && p < (int)(gridDim.x / (8 * SHARE)) * 8 * SHARE) {
    const int q = p / (8 * SHARE), r = p % (8 * SHARE);
    p = (q * 8 + (r & 7)) * SHARE + (r >> 3);
  }
  const int n0 = p * C;
  for (int u = threadIdx.x; u < units; u += 1024)
    panel[u] = *(const uint4_t*)(qweight + (size_t)(u / UPR) * N + n0 + (u % UPR) * 4);
  __syncthreads();
  for (int u = threadIdx.x; u < units; u += 1024) {
    const int r = u / UPR, c = u % UPR;
    const uint4_t p0 = *(const uint4_t*)(perm + 8 * r), p1 = *(const uint4_t*)(perm + 8 * r + 4);
    const uint32_t idx[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
    uint4_t o = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int src = min(max((int)idx[i], 0), K - 1);  // a bad index reads a wrong row, never outside
      const uint4_t w = panel[(src >> 3) * UPR + c];
      const uint32_t sh = (uint32_t)(src & 7) * 4u;
      o.x |= __builtin_amdgcn_ubfe(w.x, sh, 4u) << (4 * i);
      o.y |= __builtin_amdgcn_ubfe(w.y, sh, 4u) << (4 * i);
      o.z |= __builtin_amdgcn_ubfe(w.z, sh, 4u) << (4 * i);
      o.w |= __builtin_amdgcn_ubfe(w.w, sh, 4u) << (4 * i);
    }
    *(uint4_t*)(out + (size_t)r * N + n0 + 4 * c) = o;
  }
}

// out[m][i] = x[m][perm[i]] for 16-bit elements.  A thread gathers eight neighbours of the output
// row (one 16-byte store); the reads hit a row of x that stays in L2.
__global__ __launch_bounds__(256) void gather_columns_kernel(const uint16_t* __restrict__ x,
                                                             const int32_t* __restrict__ perm,
                                                             uint16_t* __restrict__ out, int M, int K) {
  const int vec_per_row = K >> 3;
  const long total = (long)M * vec_per_row;
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < total; v += (long)gridDim.x * blockDim.x) {
    const long m = v / vec_per_row;
    const int c = (int)(v - m * vec_per_row) * 8;
    const uint16_t* row = x + (size_t)m * K;
    const uint4_t p0 = *(const uint4_t*)(perm + c);
    const uint4_t p1 = *(const uint4_t*)(perm + c + 4);
    const uint32_t idx[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = row[min(max((int)idx[i], 0), K - 1)];
    uint4_t o;
    o.x = h[0] | (h[1] << 16);
    o.y = h[2] | (h[3] << 16);
    o.z = h[4] | (h[5] << 16);
    o.w = h[6] | (h[7] << 16);
    *(uint4_t*)(out + (size_t)m * K + c) = o;
  }
}

// Grouped form: sorted row r of expert e (offsets[e] <= r < offsets[e + 1]) becomes
// x[x_rows ? x_rows[r] : r][perms[e][.]].  Output [pairs, K] in sorted order.
__global__ __launch_bounds__(256) void moe_gather_columns_kernel(const uint16_t* __restrict__ x,
                                                                 const int32_t* __restrict__ x_rows,
                                                                 const int32_t* __restrict__ offsets,
                                                                 const int32_t* __restrict__ perms,
                                                                 uint16_t* __restrict__ out, int num_experts,
                                                                 int pairs, int K) {
  const int vec_per_row = K >> 3;
  const long total = (long)pairs * vec_per_row;
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < total; v += (long)gridDim.x * blockDim.x) {
    const int r = (int)(v / vec_per_row);
    const int c = (int)(v - (long)r * vec_per_row) * 8;
    int lo = 0, hi = num_experts;  // expert of row r: the last e with offsets[e] <= r
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (offsets[mid] <= r) lo = mid; else hi = mid;
    }
    const uint16_t* row = x + (size_t)(x_rows != nullptr ? x_rows[r] : r) * K;
    const int32_t* perm = perms + (size_t)lo * K;
    const uint4_t p0 = *(const uint4_t*)(perm + c);
    const uint4_t p1 = *(const uint4_t*)(perm + c + 4);
    const uint32_t idx[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = row[min(max((int)idx[i], 0), K - 1)];
    uint4_t o;
    o.x = h[0] | (h[1] << 16);
    o.y = h[2] | (h[3] << 16);
    o.z = h[4] | (h[5] << 16);
    o.w = h[6] | (h[7] << 16);
    *(uint4_t*)(out + (size_t)r * K + c) = o;
  }
}

// Many rows: a workgroup stages one row of x in LDS with 16-byte loads and gathers from there,
// so that global memory sees only coalesced traffic (the direct kernels above read 2-byte
// elements scattered over the row).  perms == one permutation when offsets is nullptr.
__global__ __launch_bounds__(256) void gather_rows_lds_kernel(const uint16_t* __restrict__ x,
                                                              const int32_t* __restrict__ x_rows,
                                                              const int32_t* __restrict__ offsets,
                                                              const int32_t* __restrict__ perms,
                                                              uint16_t* __restrict__ out, int num_experts, int rows,
                                                              int K) {
  extern __shared__ __align__(16) uint16_t row_lds[];  // [K]
  const int vec_per_row = K >> 3;
  for (int r = blockIdx.x; r < rows; r += gridDim.x) {
    const int32_t* perm = perms;
    if (offsets != nullptr) {
      int lo = 0, hi = num_experts;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (offsets[mid] <= r) lo = mid; else hi = mid;
      }
      perm += (size_t)lo * K;
    }
    const uint16_t* src = x + (size_t)(x_rows != nullptr ? x_rows[r] : r) * K;
    for (int v = threadIdx.x; v < vec_per_row; v += 256) ((uint4_t*)row_lds)[v] = ((const uint4_t*)src)[v];
    __syncthreads();
    for (int v = threadIdx.x; v < vec_per_row; v += 256) {
      const uint4_t p0 = *(const uint4_t*)(perm + v * 8);
      const uint4_t p1 = *(const uint4_t*)(perm + v * 8 + 4);
      const uint32_t idx[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
      uint32_t h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) h[i] = row_lds[min(max((int)idx[i], 0), K - 1)];
      uint4_t o;
      o.x = h[0] | (h[1] << 16);
      o.y = h[2] | (h[3] << 16);
      o.z = h[4] | (h[5] << 16);
      o.w = h[6] | (h[7] << 16);
      ((uint4_t*)(out + (size_t)r * K))[v] = o;
    }
    __syncthreads();
  }
}

}  // namespace q4

namespace q4host {

// rows from which the LDS-staged kernel is used (fewer rows leave most CUs without a workgroup)
static constexpr int kGatherLdsRows = 128;

static bool launch_gather_lds(const void* x, const int32_t* x_rows, const int32_t* offsets, const int32_t* perms,
                              void* out, int num_experts, int rows, int K, hipStream_t stream) {
  const size_t smem = (size_t)K * 2;
  if (rows < kGatherLdsRows || smem > 64 * 1024) return false;
  const int blocks = rows < 2048 ? rows : 2048;
  hipLaunchKernelGGL(q4::gather_rows_lds_kernel, dim3((unsigned)blocks), dim3(256), smem, stream, (const uint16_t*)x,
                     x_rows, offsets, perms, (uint16_t*)out, num_experts, rows, K);
  return true;
}


int launch_moe_gather_columns(const void* x, const int32_t* x_rows, const int32_t* offsets, const int32_t* perms,
                              void* out, int num_experts, int pairs, int K, hipStream_t stream) {
  const long total = (long)pairs * (K / 8);
  long blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) blocks = 1;
  if (!launch_gather_lds(x, x_rows, offsets, perms, out, num_experts, pairs, K, stream)) {
    hipLaunchKernelGGL(q4::moe_gather_columns_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                       (const uint16_t*)x, x_rows, offsets, perms, (uint16_t*)out, num_experts, pairs, K);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_moe_gather_columns: launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}


int launch_make_sequential(const uint32_t* qweight, const int32_t* perm, uint32_t* out, int K, int N,
                           hipStream_t stream) {
  dim3 grid((unsigned)((N + 255) / 256), (unsigned)(K / 8));
  hipLaunchKernelGGL(q4::make_sequential_kernel, grid, dim3(256), 0, stream, qweight, perm, out, K, N);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_gptq_make_sequential: launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

static constexpr size_t kRegroupLdsBytes = 150 * 1024;
// Columns of a panel, 0 when none fits LDS: 32 (one cache line a row) while that leaves a panel per CU, 16
// on narrower matrices, 8 where K asks for it (us at 32 / 16 / 8 columns: 8192 x 57344 131 / 145 / 191,
// 4096 x 28672 32.1 / 38.6 / 48.6, but 4096 x 4096 8.1 / 6.6 / 6.4).
static int regroup_panel(int K, int N) {
  for (int c = N >= 32 * 256 ? 32 : 16; c >= 8; c >>= 1)
    if ((size_t)K * c / 2 <= kRegroupLdsBytes && N % c == 0) return c;
  return 0;
}
bool regroup_supported(int K, int N) { return K % 8 == 0 && regroup_panel(K, N) != 0; }

int launch_group_order(const int32_t* g_idx, int32_t* perm, int32_t* uneven, int K, int num_groups, int groupsize,
                       hipStream_t stream) {
  hipLaunchKernelGGL(q4::group_order_kernel, dim3((unsigned)num_groups), dim3(512), 0, stream, g_idx, perm, uneven, K, groupsize);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_linear_regroup: launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

int launch_regroup(const uint32_t* qweight, const int32_t* perm, const int32_t* uneven, int num_groups, int32_t* any_uneven,
                   uint32_t* out, int K, int N, hipStream_t stream) {
  const int c = regroup_panel(K, N);
  const size_t smem = (size_t)K * c / 2;
  const dim3 grid((unsigned)(N / (c > 0 ? c : 1)));
  auto launch = [&](auto k) {
    if (smem > 64 * 1024) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipLaunchKernelGGL(k, grid, dim3(1024), smem, stream, qweight, perm, uneven, num_groups, any_uneven, out, K, N);
  };
  if (c == 32) launch(q4::regroup_kernel<32>);
  else if (c == 16) launch(q4::regroup_kernel<16>);
  else if (c == 8) launch(q4::regroup_kernel<8>);
  else {
    set_error("q4_linear_regroup: K=%d N=%d has no panel that fits LDS", K, N);
    return Q4_ERR_UNSUPPORTED;
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_linear_regroup: launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

int launch_gather_columns(const void* x, const int32_t* perm, void* out, int M, int K, hipStream_t stream) {
  const long total = (long)M * (K / 8);
  long blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) blocks = 1;
  if (!launch_gather_lds(x, nullptr, nullptr, perm, out, 1, M, K, stream)) {
    hipLaunchKernelGGL(q4::gather_columns_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint16_t*)x,
                       perm, (uint16_t*)out, M, K);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("q4_gather_columns: launch failed: %s", hipGetErrorString(err));
    return Q4_ERR_LAUNCH;
  }
  return Q4_OK;
}

}  // namespace q4host

// Products of a few rows with weight matrices, y = x W^T: a decode step's
// projections (src/lizard_attention.py:73-76,97 at one token per sequence).
//
// Up to 16 rows x [M, K] bf16 against up to four matrices W [N_i, K] bf16 in one
// launch, fp32 sums, rounded to bf16 once.  The weights' bytes are all there is to
// it, each read once: a workgroup takes 16 rows of one matrix, its eight waves
// interleaved pieces of K (64 columns a step, four steps' loads in flight), as
// 16x16x32 MFMA tiles (A = 16 weight rows, B = the M rows, zero past M); the
// waves' partial tiles meet in LDS and are added in wave order.  Within a step a
// lane's 16 columns are consecutive, so a row is read in whole 128-byte lines;
// which k index an operand slot carries is free as long as A and B agree.
// Measured at hidden 2048 with 32/8 heads, 4 rows: q, k, v and the gate (12.6 MB)
// 7.2 us and o_proj (8.4 MB) 5.2 us, launched back to back, where the library's products took 29 and
// 8.4 us of GPU time and 83 us of host time for choosing them.
#include "common.hpp"

namespace lz {

constexpr int ROWS_MATS = 4;   // LZ_ROWS_MATS
constexpr int ROWS_WAVES = 8, ROWS_STEP = 64, ROWS_BATCH = 4;

// blk0: the first workgroup of a matrix; f32: y in fp32 (of the bf16 result)
struct RowsMats {
  const bf16* w[ROWS_MATS];
  void* y[ROWS_MATS];
  int n[ROWS_MATS], blk0[ROWS_MATS], f32[ROWS_MATS];
};

__global__ __launch_bounds__(64 * ROWS_WAVES) void rows_linear_kernel(
    const bf16* __restrict__ x, int M, int K, int mats, RowsMats m) {
  __shared__ float red[ROWS_WAVES][16][17];
  int i = 0;
#pragma unroll
  for (int j = 1; j < ROWS_MATS; ++j)
    if (j < mats && (int)blockIdx.x >= m.blk0[j]) i = j;
  const int n = m.n[i], n0 = 16 * ((int)blockIdx.x - m.blk0[i]);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  // rows past a matrix's last lie past its resource, as do x rows past M
  const rsrc_t wr = make_rsrc(m.w[i], (size_t)n * K * 2);
  const rsrc_t xr = make_rsrc(x, (size_t)M * K * 2);
  const int steps = (K + ROWS_STEP - 1) / ROWS_STEP;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = wave; s0 < steps; s0 += ROWS_WAVES * ROWS_BATCH) {
    bf16x8 a[ROWS_BATCH][2], b[ROWS_BATCH][2];
#pragma unroll
    for (int t = 0; t < ROWS_BATCH; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = ROWS_STEP * (s0 + ROWS_WAVES * t) + 16 * g + 8 * e;   // K % 8 == 0
        const bool in = k < K;
        a[t][e] = __builtin_bit_cast(
            bf16x8, bload16<LOAD_NT>(wr, in ? (uint32_t)((n0 + col) * K + k) * 2u : OOB));
        b[t][e] = __builtin_bit_cast(bf16x8, bload16(xr, in ? (uint32_t)(col * K + k) * 2u : OOB));
      }
#pragma unroll
    for (int t = 0; t < ROWS_BATCH; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][e], b[t][e], acc, 0, 0, 0);
  }
  // lane: column (x row) col, weight rows 4 g + r
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][4 * g + r][col] = acc[r];
  __syncthreads();
  const int row = threadIdx.x & 15, xi = threadIdx.x >> 4;   // the first 256 threads
  if (xi < M && n0 + row < n) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < ROWS_WAVES; ++w) sum += red[w][row][xi];
    const bf16 out = to_bf16(sum);
    const size_t at = (size_t)xi * n + n0 + row;
    if (m.f32[i])
      static_cast<float*>(m.y[i])[at] = to_f32(out);
    else
      static_cast<bf16*>(m.y[i])[at] = out;
  }
}

hipError_t launch_rows_linear(const void* x, int M, int K, int mats, const void* const* w,
                              void* const* y, const int* n, const int* f32, hipStream_t st) {
  RowsMats m = {};
  int blocks = 0;
  for (int i = 0; i < mats; ++i) {
    m.w[i] = (const bf16*)w[i];
    m.y[i] = y[i];
    m.n[i] = n[i];
    m.f32[i] = f32[i];
    m.blk0[i] = blocks;
    blocks += (n[i] + 15) / 16;
  }
  hipLaunchKernelGGL(rows_linear_kernel, dim3(blocks), dim3(64 * ROWS_WAVES), 0, st,
                     (const bf16*)x, M, K, mats, m);
  return hipGetLastError();
}

}  // namespace lz

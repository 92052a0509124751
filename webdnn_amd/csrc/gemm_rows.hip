// Products of a few rows with a transposed weight, Y[m, n] = A[m, k] . W[n, k]^T for m <= 4 (a request through a
// fully connected net, the classifier of one picture).
//
// Bound: reading W once.  The 32-row matrix-core blocks of gemm_wavesplit_kernel multiply 28 to 31 rows of padding
// and fetch W in 64-byte pieces of 32 different rows; here a wavefront reads whole rows of W, 1 KB an instruction,
// and keeps the sums in registers.  A wavefront owns two columns (rows of W), so that a piece of A is loaded once
// for two pieces of W, four steps (8 KB of W) in flight; where n leaves fewer than eight wavefronts a CU
// the four wavefronts of a workgroup share K instead and meet in LDS.  Sums are fp32, a lane's share of K in
// index order and then a fixed tree over the lanes, so results do not depend on scheduling.
//
// One row, replayed (us; gemm_wavesplit_kernel or cut 64x64 tiles before -> now): n 4096, k 4096 28.5 -> 13.4;
// 8192, 8192 62.4 -> 46.4 (5.8 TB/s); 1000, 4096 20.2 -> 4.8; 10, 4096 14.4 -> 2.5; 256, 256 3.5 -> 2.4.
#include "contraction.h"

namespace {
using namespace wdhc;

constexpr int ROWS_WAVES = 4;  // wavefronts of a workgroup
constexpr int ROWS_COLS = 2;   // columns of a wavefront

template <int M, bool VEC, bool SHARE_K>
__global__ __launch_bounds__(64 * ROWS_WAVES) void gemm_rows_kernel(Params p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col0 = ((int)blockIdx.x * (SHARE_K ? 1 : ROWS_WAVES) + (SHARE_K ? 0 : wave)) * ROWS_COLS;
  const long long bz = blockIdx.y;
  const float *A = p.A + bz * p.sAb;
  const float *B[ROWS_COLS];
#pragma unroll
  for (int c = 0; c < ROWS_COLS; c++)  // (columns past the edge read the last one and are not stored)
    B[c] = p.B + bz * p.sBb + (long long)(col0 + c < p.n ? col0 + c : p.n - 1) * p.sB1;
  float acc[M][ROWS_COLS];
#pragma unroll
  for (int r = 0; r < M; r++)
#pragma unroll
    for (int c = 0; c < ROWS_COLS; c++) acc[r][c] = 0.0f;

  const int part = (SHARE_K ? wave * 64 : 0) + lane;
  constexpr int STEP = 64 * (SHARE_K ? ROWS_WAVES : 1);  // lanes that walk K together
  const int whole = VEC ? p.k / 4 : 0;                   // 16-byte pieces of a row
  constexpr int U = 4;
  int q = part;
  auto add = [&](int piece, const f32x4 (&b)[ROWS_COLS]) {
#pragma unroll
    for (int r = 0; r < M; r++) {
      const f32x4 a = reinterpret_cast<const f32x4 *>(A + r * p.sA0)[piece];
#pragma unroll
      for (int c = 0; c < ROWS_COLS; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[r][c] = __builtin_fmaf(a[e], b[c][e], acc[r][c]);
    }
  };
  if (VEC) {
    // (the lanes that share K leave this loop together: where some still have U pieces and others do not, the wavefront
    // pays for both loops; 3 rows, n 8192, k 1000 11.4 -> 7.9 us, and k 800, 3000, 6000 are back ahead of the other form)
    const int end = whole - whole % (U * STEP);
    for (; q < end; q += U * STEP) {
      f32x4 b[U][ROWS_COLS];
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int c = 0; c < ROWS_COLS; c++) b[u][c] = reinterpret_cast<const f32x4 *>(B[c])[q + u * STEP];
#pragma unroll
      for (int u = 0; u < U; u++) add(q + u * STEP, b[u]);
    }
    for (; q < whole; q += STEP) {
      f32x4 b[ROWS_COLS];
#pragma unroll
      for (int c = 0; c < ROWS_COLS; c++) b[c] = reinterpret_cast<const f32x4 *>(B[c])[q];
      add(q, b);
    }
  }
  // rows that are not 16-byte aligned, and what a row holds beyond its whole pieces
  for (int x = 4 * whole + part; x < p.k; x += STEP)
#pragma unroll
    for (int r = 0; r < M; r++)
#pragma unroll
      for (int c = 0; c < ROWS_COLS; c++) acc[r][c] = __builtin_fmaf(A[r * p.sA0 + x], B[c][x], acc[r][c]);

#pragma unroll
  for (int r = 0; r < M; r++)
#pragma unroll
    for (int c = 0; c < ROWS_COLS; c++)
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) acc[r][c] += __shfl_xor(acc[r][c], d);

  // lane i of the (first) wavefront finishes result i of the M x 2
  float sum = acc[0][0];
#pragma unroll
  for (int r = 0; r < M; r++)
#pragma unroll
    for (int c = 0; c < ROWS_COLS; c++)
      if (lane == r * ROWS_COLS + c) sum = acc[r][c];
  if (SHARE_K) {
    __shared__ float parts[ROWS_WAVES][M * ROWS_COLS];
    if (lane < M * ROWS_COLS) parts[wave][lane] = sum;
    __syncthreads();
    if (wave != 0) return;
    sum = parts[0][lane < M * ROWS_COLS ? lane : 0];
#pragma unroll
    for (int w = 1; w < ROWS_WAVES; w++) sum += parts[w][lane < M * ROWS_COLS ? lane : 0];
  }
  const int row = lane / ROWS_COLS, col = col0 + lane % ROWS_COLS;
  if (row >= M || col >= p.n) return;
  float y = p.alpha * sum;
  if (p.C) y = __builtin_fmaf(p.C[(long long)row * p.sC0 + (long long)col * p.sC1], p.beta, y);
  const long long off = bz * p.sYb + (long long)row * p.sY0 + col;
  if (p.R) y = y + p.R[off];
  if (p.epilogue == WDH_EPI_RELU) y = relu_js(y);
  p.Y[off] = y;
}

template <int M>
void start(const Params &p, int batch, bool vec, bool share) {
  const int cols = share ? ROWS_COLS : ROWS_COLS * ROWS_WAVES;
  const dim3 grid((unsigned)(((long long)p.n + cols - 1) / cols), (unsigned)batch), block(64 * ROWS_WAVES);
  if (vec && share) hipLaunchKernelGGL((gemm_rows_kernel<M, true, true>), grid, block, 0, wdh::stream(), p);
  else if (vec) hipLaunchKernelGGL((gemm_rows_kernel<M, true, false>), grid, block, 0, wdh::stream(), p);
  else if (share) hipLaunchKernelGGL((gemm_rows_kernel<M, false, true>), grid, block, 0, wdh::stream(), p);
  else hipLaunchKernelGGL((gemm_rows_kernel<M, false, false>), grid, block, 0, wdh::stream(), p);
}
}  // namespace

namespace wdhc {
long long gemm_rows_waves(int n, int batch) { return ((long long)n + ROWS_COLS - 1) / ROWS_COLS * batch; }
// Fewer than eight wavefronts a CU leave too few loads in flight: the four of a workgroup then share K.
bool gemm_rows_share_k(long long waves) { return waves < 8LL * wdh::compute_units(); }

// A and B k-contiguous, 1 <= m <= GEMM_ROWS_MAX; vec: bases and strides keep 16-byte alignment.
int launch_gemm_rows(const Params &p, int batch, bool vec) {
  const long long waves = gemm_rows_waves(p.n, batch);
  const bool share = gemm_rows_share_k(waves);
  switch (p.m) {
    case 1: start<1>(p, batch, vec, share); break;
    case 2: start<2>(p, batch, vec, share); break;
    case 3: start<3>(p, batch, vec, share); break;
    default: start<4>(p, batch, vec, share); break;
  }
  g_last_plan = {p.m, ROWS_COLS, share ? ROWS_WAVES : 1, WDH_FORM_GEMM_KC, waves, 0};
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}
}  // namespace wdhc

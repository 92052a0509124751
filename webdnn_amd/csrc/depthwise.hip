// Depthwise 2-D convolution (one input channel per group), NCHW, bias / residual / Relu in the epilogue.
//
// Semantics: src/descriptor_runner/operators/cpu/operators/standard/conv.ts:134-333 with group = channels.
//
// A depthwise convolution is K*K multiplications per output and no contraction over channels, so the
// matrix-core kernels spend a 64-row tile on its one row per group.  Here it is what it is bound by, a
// pass over memory: a thread owns 4 neighbouring columns of ROWS output rows of one plane,
// reads the input rows they touch with one or two 16-byte loads plus the columns that stick out on either
// side, and keeps everything in registers; the rows shared by neighbouring threads come from the vector
// L1.  Threads are numbered through all planes (columns fastest), so planes of 7x7 pack into wavefronts as
// well as planes of 112x112.
// Measured (us, graph replays, batch 8, against the gathered 64x64 tiles): 3x3 32 @112x112 163.7 -> 10.7
// (25.7 MB, 2.4 TB/s), 3x3 stride 2 64 @112x112 85.5 -> 7.3 (4.4 TB/s), 3x3 512 @14x14 46.6 -> 5.6,
// 3x3 1024 @7x7 27.5 -> 4.6, 5x5 256 @28x28 130.5 -> 14.3; batch 1, 3x3 32 @112x112 24.5 -> 3.5.
#include "common.h"
#include "fastdiv.h"

namespace {

using wdh::FastDiv;
using wdh::fdiv;
using wdh::make_fastdiv;

// (16-byte accesses at 4-byte aligned addresses: rows of any length)
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4u __attribute__((aligned(4)));

struct DwParams {
  const float *X, *W, *Bias, *R;
  float *Y;
  int h, w, oh, ow, cout, mult;   // mult: output channels per input channel
  int pt, pl, kh, kw, sh, sw, dh, dw, relu;
  unsigned total;                 // work items (threads with something to do)
  FastDiv fd_tiles_x, fd_tiles, fd_cout, fd_mult;
  int tiles_x, tiles;             // 4-column tiles per row; tiles per plane
};

__device__ __forceinline__ float finish(const DwParams &p, float v, float bias, const float *r) {
  v = v + bias;
  if (r) v = v + *r;
  // Math.max(v, 0): NaN stays NaN, -0 becomes +0
  return p.relu ? (v <= 0.0f ? 0.0f : v) : v;
}

// K x K taps, stride S in both directions, left padding (K-1)/2, no dilation.
template <int K, int S, int ROWS>
__global__ __launch_bounds__(256) void depthwise_tile_kernel(DwParams p) {
  const unsigned id = blockIdx.x * 256u + threadIdx.x;
  if (id >= p.total) return;
  const int plane = fdiv((int)id, p.fd_tiles);                  // (image, output channel)
  const int tile = (int)id - plane * p.tiles;
  const int ty = fdiv(tile, p.fd_tiles_x), tx = tile - ty * p.tiles_x;
  const int img = fdiv(plane, p.fd_cout), oc = plane - img * p.cout;
  const int in_plane = img * (p.cout / p.mult) + (p.mult == 1 ? oc : fdiv(oc, p.fd_mult));
  const float *x = p.X + (long long)in_plane * p.h * p.w;
  constexpr int PL = (K - 1) / 2;
  constexpr int MID = 4 * S;                                    // columns read 16 bytes at a time
  constexpr int SPAN = 3 * S + K;                               // columns the four outputs touch
  constexpr int RIGHT = SPAN - PL - MID > 0 ? SPAN - PL - MID : 0;
  constexpr int INROWS = (ROWS - 1) * S + K;
  const int oy0 = ty * ROWS, ox0 = tx * 4;
  const int iy0 = oy0 * S - p.pt, ix0 = ox0 * S;                // ix0: first of the 16-byte columns

  float wt[K * K];
#pragma unroll
  for (int i = 0; i < K * K; i++) wt[i] = p.W[oc * (K * K) + i];
  const float bias = p.Bias ? p.Bias[oc] : 0.0f;

  float v[INROWS][PL + MID + RIGHT];
  const bool whole = ix0 + MID <= p.w;
#pragma unroll
  for (int r = 0; r < INROWS; r++) {
    const int iy = iy0 + r;
    const bool row_in = (unsigned)iy < (unsigned)p.h;
    const float *row = x + (row_in ? iy : 0) * p.w;             // (taps in the padding read row 0 and count as 0)
#pragma unroll
    for (int c = 0; c < PL; c++) {
      const int ix = ix0 - PL + c;
      const float t = row[ix >= 0 ? (ix < p.w ? ix : p.w - 1) : 0];
      v[r][c] = row_in && ix >= 0 && ix < p.w ? t : 0.0f;
    }
    if (whole) {
#pragma unroll
      for (int q = 0; q < S; q++) {
        const f32x4 t = *reinterpret_cast<const f32x4u *>(row + ix0 + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; e++) v[r][PL + 4 * q + e] = row_in ? t[e] : 0.0f;
      }
    } else {
#pragma unroll
      for (int c = 0; c < MID; c++) {
        const int ix = ix0 + c;
        const float t = row[ix < p.w ? ix : p.w - 1];
        v[r][PL + c] = row_in && ix < p.w ? t : 0.0f;
      }
    }
#pragma unroll
    for (int c = 0; c < RIGHT; c++) {
      const int ix = ix0 + MID + c;
      const float t = row[ix < p.w ? ix : p.w - 1];
      v[r][PL + MID + c] = row_in && ix < p.w ? t : 0.0f;
    }
  }
  const long long out_plane = (long long)plane * p.oh * p.ow;
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    const int oy = oy0 + r;
    if (oy >= p.oh) break;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ky = 0; ky < K; ky++)
#pragma unroll
      for (int kx = 0; kx < K; kx++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(v[r * S + ky][e * S + kx], wt[ky * K + kx], acc[e]);
    const long long off = out_plane + (long long)oy * p.ow + ox0;
    if (ox0 + 4 <= p.ow) {
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] = finish(p, acc[e], bias, p.R ? p.R + off + e : nullptr);
      *reinterpret_cast<f32x4u *>(p.Y + off) = y;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (ox0 + e < p.ow) p.Y[off + e] = finish(p, acc[e], bias, p.R ? p.R + off + e : nullptr);
    }
  }
}

// Any other kernel size, stride, padding or dilation: a thread per output, taps from the vector L1.
__global__ __launch_bounds__(256) void depthwise_any_kernel(DwParams p) {
  const unsigned id = blockIdx.x * 256u + threadIdx.x;
  if (id >= p.total) return;
  const int plane = fdiv((int)id, p.fd_tiles);
  const int cell = (int)id - plane * p.tiles;
  const int oy = fdiv(cell, p.fd_tiles_x), ox = cell - oy * p.tiles_x;
  const int img = fdiv(plane, p.fd_cout), oc = plane - img * p.cout;
  const int in_plane = img * (p.cout / p.mult) + (p.mult == 1 ? oc : fdiv(oc, p.fd_mult));
  const float *x = p.X + (long long)in_plane * p.h * p.w;
  const float *w = p.W + (long long)oc * p.kh * p.kw;
  float acc = 0.0f;
  for (int ky = 0; ky < p.kh; ky++) {
    const int iy = oy * p.sh - p.pt + ky * p.dh;
    const bool row_in = (unsigned)iy < (unsigned)p.h;
    for (int kx = 0; kx < p.kw; kx++) {
      const int ix = ox * p.sw - p.pl + kx * p.dw;
      const bool in = row_in && (unsigned)ix < (unsigned)p.w;
      const float t = x[in ? (long long)iy * p.w + ix : 0];
      acc = __builtin_fmaf(in ? t : 0.0f, w[ky * p.kw + kx], acc);
    }
  }
  const long long off = (long long)plane * p.oh * p.ow + cell;
  p.Y[off] = finish(p, acc, p.Bias ? p.Bias[oc] : 0.0f, p.R ? p.R + off : nullptr);
}

template <int K, int S, int ROWS>
void start(const DwParams &p) {
  hipLaunchKernelGGL((depthwise_tile_kernel<K, S, ROWS>), dim3((p.total + 255u) / 256u), dim3(256), 0, wdh::stream(), p);
}

}  // namespace

namespace wdh {

bool depthwise_applies(int n, int cout, int c_in_g, int cout_g, int group, int oh, int ow) {
  // The thread numbering is 32-bit.  Many output channels per input channel are a product again: 64 channels
  // @56x56, batch 8, take 11.0 / 13.6 / 23.8 / 42.4 us here with 2 / 4 / 8 / 16 outputs each and 85 / 86 / 88 / 93
  // as 64-row tiles, which cost the same up to 64 outputs; past 16 the two meet.
  return c_in_g == 1 && cout_g <= 16 && (long long)n * cout * oh * ow <= 0x7fffffffLL - 256 &&
         (long long)n * group < 0x7fffffffLL;
}

int depthwise_launch(const float *X, const float *W, const float *Bias, const float *R, float *Y, int n, int c, int h,
                     int w, int cout, int kh, int kw, int pt, int pl, int sh, int sw, int dh, int dw, int oh, int ow,
                     int relu, DepthwisePlan &plan) {
  DwParams p = {};
  p.X = X; p.W = W; p.Bias = Bias; p.R = R; p.Y = Y;
  p.h = h; p.w = w; p.oh = oh; p.ow = ow; p.cout = cout; p.mult = cout / c;
  p.pt = pt; p.pl = pl; p.kh = kh; p.kw = kw; p.sh = sh; p.sw = sw; p.dh = dh; p.dw = dw; p.relu = relu;
  p.fd_cout = make_fastdiv(cout);
  p.fd_mult = make_fastdiv(p.mult);
  const long long planes = (long long)n * cout;
  auto tiled = [&](int rows, int cols) {
    p.tiles_x = (ow + cols - 1) / cols;
    p.tiles = p.tiles_x * ((oh + rows - 1) / rows);
    p.fd_tiles_x = make_fastdiv(p.tiles_x);
    p.fd_tiles = make_fastdiv(p.tiles);
    p.total = (unsigned)(planes * p.tiles);
  };
  const bool tile = kh == kw && sh == sw && dh == 1 && dw == 1 && pl == (kw - 1) / 2 && (kh == 3 || kh == 5) && sh <= 2;
  if (!tile) {
    tiled(1, 1);
    plan = {1, 1, planes * p.tiles};
    hipLaunchKernelGGL(depthwise_any_kernel, dim3((p.total + 255u) / 256u), dim3(256), 0, wdh::stream(), p);
    WDH_LAUNCH_CHECK();
    return WDH_OK;
  }
  // Several rows per thread read the shared input rows once; below four threads per lane of the chip
  // it pays more to have every SIMD busy.
  const int rows = sh == 1 ? 4 : 2;
  const bool tall = planes * ((ow + 3) / 4) * ((oh + rows - 1) / rows) >= 4LL * 64 * 4 * compute_units();
  tiled(tall ? rows : 1, 4);
  plan = {tall ? rows : 1, 4, planes * p.tiles};
  if (kh == 3 && sh == 1) tall ? start<3, 1, 4>(p) : start<3, 1, 1>(p);
  else if (kh == 3) tall ? start<3, 2, 2>(p) : start<3, 2, 1>(p);
  else if (sh == 1) tall ? start<5, 1, 4>(p) : start<5, 1, 1>(p);
  else tall ? start<5, 2, 2>(p) : start<5, 2, 1>(p);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}

}  // namespace wdh

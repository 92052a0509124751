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

// Any other kernel size, stride, padding or dilation, and small launches: a thread per output, taps from the vector L1.
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
  // (a sum a row of the kernel, since rounding errors grow with the length of a chain: 31x31, 128 channels @28x28, 2-norm
  // error against 64 bits 1.3e-7, 4.15e-7 as one chain and 4.08e-7 as matrix tiles cut in two along the taps)
  float acc = 0.0f;
  for (int ky = 0; ky < p.kh; ky++) {
    const int iy = oy * p.sh - p.pt + ky * p.dh;
    const bool row_in = (unsigned)iy < (unsigned)p.h;
    float row = 0.0f;
    for (int kx = 0; kx < p.kw; kx++) {
      const int ix = ox * p.sw - p.pl + kx * p.dw;
      const bool in = row_in && (unsigned)ix < (unsigned)p.w;
      const float t = x[in ? (long long)iy * p.w + ix : 0];
      row = __builtin_fmaf(in ? t : 0.0f, w[ky * p.kw + kx], row);
    }
    acc += row;
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

// The geometries depthwise_tile_kernel is built for.
static bool tile_geometry(int kh, int kw, int pl, int sh, int sw, int dh, int dw) {
  return kh == kw && sh == sw && dh == 1 && dw == 1 && pl == (kw - 1) / 2 && (kh == 3 || kh == 5) && sh <= 2;
}
// Rows whose last tile is ragged take both paths of the tile kernel, load by load.  Up to 512 outputs a CU that
// latency is all of the time, and a thread per output is done sooner (us, tile against cell kernel, 7x7 planes): 3x3
// 4.7 / 3.9, stride 2 5.6 / 4.0, 5x5 6.7 / 5.3, stride 2 8.2 / 5.4; from twice as many outputs on the tiles are ahead.
static bool tile_suits(long long outputs, int ow) { return ow % 4 == 0 || outputs > 512LL * compute_units(); }
// Several rows per thread read the shared input rows once; below four threads per lane of the chip it pays more to
// have every SIMD busy (us, one row a thread against several): 3x3 32 @112x112 batch 4 / 8 / 16 / 32 6.9 / 11.8 / 20.0 /
// 36.5 against 7.6 / 10.6 / 14.3 / 26.4, 5x5 16.2 / 26.2 / 46.6 / 85.6 against 11.8 / 17.4 / 29.8 / 55.2; 3x3 stride 2
// gains or loses 5 %; 3x3 512 @14x14, where every fourth row of the tiles is empty, batch 64 25.2 against 34.8.
static bool several_rows(long long planes, int sh, int oh, int ow) {
  const int rows = sh == 1 ? 4 : 2;
  return planes * ((ow + 3) / 4) * ((oh + rows - 1) / rows) >= 4LL * 64 * 4 * compute_units();
}

bool depthwise_fits(int n, int cout, int c_in_g, int cout_g, int group, int oh, int ow) {
  // (the thread numbering is 32-bit)
  return c_in_g == 1 && cout_g <= 16 && (long long)n * cout * oh * ow <= 0x7fffffffLL - 256 && (long long)n * group < 0x7fffffffLL;
}

// Whether the pass over memory beats the gathered matrix tiles, by an estimate of both (us), fitted to a sweep of 6900
// geometries: 1x1 to 31x31 taps, planes of 1 to 112x112, 1 to 1024 channels of 1 to 16 outputs, batch 1 to 64.  Both
// sides measured there, it takes the pass where that is 4 to 7 % slower in 18 of them, and leaves 246 to the tiles that
// the pass would do in 0.7 to 0.96 of the time (two in 0.54), sixteen outputs a channel or planes of a few cells mostly.
bool depthwise_applies(int n, int cout, int c_in_g, int cout_g, int group, int kh, int kw, int pl, int sh, int sw, int dh,
                       int dw, int oh, int ow) {
  if (!depthwise_fits(n, cout, c_in_g, cout_g, group, oh, ow)) return false;
  const double chip = compute_units() / 256.0, taps = (double)kh * kw;
  const double planes = (double)n * group, outputs = (double)n * cout * oh * ow;
  auto larger = [](double a, double b) { return a > b ? a : b; };
  // The tiles compute 64 rows for a group's one to sixteen, whatever their number, and cut long sums along the taps.
  const double tiles = (double)group * (double)(((long long)n * oh * ow + 63) / 64) / 256.0 / chip;
  const double matrix_us = 4.0 + larger(1.0 + (taps < 41.0 ? 0.12 * taps : 5.0), tiles * (0.7 + 0.022 * taps + (taps > 31.0 && taps < 64.0 ? 0.35 : 0.0)));
  // Here a tap costs every output: 3x3 dilated, 64 channels @56x56, batch 8, of 2 / 4 / 8 / 16 outputs each 26 / 45 / 81 /
  // 143 us against 85 / 87 / 87 / 91 as tiles.
  if (tile_geometry(kh, kw, pl, sh, sw, dh, dw) && tile_suits((long long)n * cout * oh * ow, ow)) {
    // [5x5][stride 2][ragged rows] ([several rows a thread]): the least time, and 10^6 outputs per us
    static const double least[2][2][2] = {{{3.9, 4.7}, {3.8, 5.6}}, {{5.3, 6.7}, {5.1, 8.2}}};
    static const double rate[2][2][2][2] = {{{{0.5, 0.5}, {0.5, 0.5}}, {{0.35, 0.35}, {0.15, 0.17}}},
                                            {{{0.18, 0.4}, {0.15, 0.4}}, {{0.16, 0.17}, {0.08, 0.115}}}};
    const int i = kh == 5, j = sh == 2, r = ow % 4 != 0;
    return larger(least[i][j][r], 2.3 + outputs / (rate[i][j][r][several_rows((long long)n * cout, sh, oh, ow)] * 1e6 * chip)) < matrix_us;
  }
  // The cell kernel: a thread's taps are one chain (a 28x28 kernel over a 28x28 plane 185 us against 30), and
  // neighbouring threads that read different planes fetch a line each.
  const int plane = oh * ow < 16 ? oh * ow : 16;
  if (plane < 4)
    return 2.3 + 0.16 * taps + planes * taps / ((taps > 9.0 ? 0.17e6 : 1e6) * chip) +
           outputs * taps / ((taps > 25.0 ? 0.4e6 : 1.2e6) * chip) < matrix_us;
  const double tap_rate = plane < 9 ? (taps > 100.0 ? 0.6e6 : 1.2e6)
                          : ow >= 32 || oh * ow % 16 == 0 ? (taps > 25.0 ? 2.3e6 : 1.8e6)
                          : ow >= 16 ? 1.8e6 : taps > 81.0 ? 1.05e6 : 1.25e6;
  return 2.3 + larger((plane < 9 ? 0.13 : taps > 49.0 ? 0.098 : 0.11) * taps, outputs / chip * larger(taps / tap_rate, 1.0 / (taps > 1.0 ? 0.2e6 : 0.3e6))) < matrix_us;
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
  if (!tile_geometry(kh, kw, pl, sh, sw, dh, dw) || !tile_suits(planes * oh * ow, ow)) {
    tiled(1, 1);
    plan = {1, 1, planes * p.tiles};
    hipLaunchKernelGGL(depthwise_any_kernel, dim3((p.total + 255u) / 256u), dim3(256), 0, wdh::stream(), p);
    WDH_LAUNCH_CHECK();
    return WDH_OK;
  }
  const int rows = sh == 1 ? 4 : 2;
  const bool tall = several_rows(planes, sh, oh, ow);
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

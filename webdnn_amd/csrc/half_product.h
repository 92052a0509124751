// Products of fp32 operands on the f16 matrix cores, at the precision of the products in bfloat16 parts (split_product.h) or better, in
// half as many matrix instructions.
//
// A float, scaled into f16's range by a power of two, is h + l / 2^11 but for its last bit: h is the nearest f16 value, l the nearest to
// 2^11 times what is left (the scaling of l keeps its bits where h is small).  Of the four products h*h, h*l and l*h go through
// v_mfma_f32_16x16x32_f16; l*l is left out.  What that costs is a floor of 1.0e-7 in the 2-norm against 64 bits (6.2e-8 the last
// bits, 4.3e-8 l*l), so the chains of additions must be the better ones: a block of 64 k starts from zero, h*h and the two small
// products in accumulators of their own, and is added to the totals by vector instructions, which round a sum less badly than the
// matrix core adds to it (K 1024 1.24e-7, 4096 1.77e-7; in bfloat16 parts 1.9e-7 and 4.0e-7).  The accumulators are needed for
// one group of two strips x 16 columns at a time, so that only the totals stay in registers.  half_is_as_precise (gemm.hip) draws the line.
//
// One operand (weights; a product's right operand) is packed beforehand, row by row scaled, in the order in which lanes want it, and
// goes from L2 straight into registers; the other is split on its way from registers to LDS, as in split_product.h.  That halves both
// the LDS traffic and the vector instructions of a version with both operands in LDS (4096^3, us: 522 so, 395 packed; and with every strip
// read by one wavefront instead of two, 32 rows x 128 columns each: 427 with packing for 455).
//
// Bound: no unit by itself.  The matrix cores are busy 0.62 of the time at 4096^3, 0.4 in 1x1 convs, the rest goes into vector
// instructions (two an element every 64 k, three an element for the split), LDS reads and waits for L2, and into a start and an end of 9 to
// 12 us, part of it code that arrives line by line; launched in a row, power joins in (415 us, the seventh 468).  A loop of nothing but the instruction makes 1830 TFLOP/s (32x32x16: 1640, bf16 16x16x32 1960), 610 of
// products; 4096^3 349 without the packing (bfloat16 parts 212), 1024 -> 256 on 14x14 with 128 images 195 (142), 128 -> 128 3x3
// on 28x28 222 (197).  Tried without gain: 64x64 a wavefront, groups of 32 columns, totals added a group later without reads ahead, LDS planes
// 16 to 64 bytes apart, two buffers of rows for 3x3 convs of 640 pixels.
//
// What the two parts cannot hold is done again with the fp32 instruction, a whole tile (or chunk) at a time:
//   * an Inf, a NaN or an element that outgrows f16 (the other operand is scaled by the largest element of a tile's first block to 2^10
//     to 2^11, which leaves a factor of 32 to 64) leaves NaN or Inf in every sum it enters;
//   * an element below 2^-13 (scaled) is off by up to 2^-36, one below 2^-36 by all of itself.  K such elements against partners of
//     up to 2^16 change a sum by K 2^-20 at most, so sums of 16 and more do not show them.  A tile with a smaller sum
//     (one in a hundred of normally distributed ones) counts those elements, column by column, and is done again if a
//     sum is smaller than 16 / K times the count of its row and column: less than one tile in 10^5, but zeros among many
//     magnitudes can come to that.
#pragma once
#include "contraction.h"

namespace wdhc {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int W_TARGET = 14, X_TARGET = 10;  // exponents that the largest of a packed row, of a tile's first block are scaled to
constexpr int W_ROOM = 3;            // less, where only the beginning of the row is known
constexpr float LOW_SCALE = 2048.0f;
constexpr int FULL_EXPONENT = -13;   // from 2^this on a scaled element keeps 23 bits; smaller ones are off by up to 2^-36
constexpr float SAFE_SUM = 16.0f;    // sums from here on (scaled) do not show what such elements lost

// Eight elements -> their two parts, scaled by `s`.  (Three instructions an element: v_fma_mixlo_f16, v_fma_mix_f32, v_fma_mixlo_f16.)
struct HalfParts { f16x8 h, l; };
__device__ __forceinline__ HalfParts half_parts(const float (&x)[8], float s) {
  HalfParts q;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const _Float16 h = (_Float16)__builtin_fmaf(x[i], s, 0.0f);
    const float r = __builtin_fmaf(x[i], s, -(float)h);
    q.h[i] = h;
    q.l[i] = (_Float16)__builtin_fmaf(r, LOW_SCALE, 0.0f);
  }
  return q;
}
// The exponent that scales magnitudes with these (absolute) bits to `target`; what cannot be scaled stays.
__host__ __device__ __forceinline__ int scale_exponent(unsigned bits, int target) {
  const int e = (int)(bits >> 23);
  if (bits == 0 || e == 255) return 0;
  const int q = target - ((e > 0 ? e : 1) - 127);
  return q < 127 ? q : 127;
}
__device__ __forceinline__ float scale_of(int exponent) { return __uint_as_float((unsigned)(exponent + 127) << 23); }

enum HalfSource { H_ROWS = 0, H_PIXELS = 1 };  // the other operand: rows of A (k-contiguous), pixels of X in place

__device__ __forceinline__ void swap16(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

// What a wavefront has of a tile: two strips of packed rows x QB columns of sixteen, [strip][columns], as
// v_mfma_f32_16x16x32_f16 leaves them.  PACKED_ROWS: the packed operand is the left one, a lane has rows 4 * (lane / 16) to + 3
// of a strip; otherwise the right one, a lane has its row lane % 16.
template <int QB> using HalfSums = f32x4[2][QB];
struct HalfDoubt { bool bad, tiny; };  // sums that are not finite; sums that might show what small elements lost
// The sums unscaled, and what they say.  (A row or a column past the edge is a zero or repeats the last: zeros raise a doubt that
// shows_loss settles.  Few instructions on purpose: a workgroup runs them once, and code that no workgroup has run yet arrives
// at 50 ns a line of 64 bytes.)
template <bool PACKED_ROWS, int QB>
__device__ __forceinline__ HalfDoubt unscale(HalfSums<QB> &sums, const HalfOperand &w, int strip0, int np, int eq) {
  const int *const exps = reinterpret_cast<const int *>(w.packed + half_fragment_bytes(w.strips, w.steps));
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  float nothing = 0.0f, least = __builtin_inff();  // (0 * Inf and 0 * NaN are NaN)
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int rows = (strip0 + i) * 16;
    if (rows >= np) break;
    int ep[PACKED_ROWS ? 4 : 1];
#pragma unroll
    for (int r = 0; r < (PACKED_ROWS ? 4 : 1); r++) ep[r] = -(exps[rows + (PACKED_ROWS ? 4 * g4 + r : c16)] + eq);
#pragma unroll
    for (int j = 0; j < QB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float v = sums[i][j][r], y = __builtin_ldexpf(v, ep[PACKED_ROWS ? r : 0]);
        least = __builtin_fminf(least, __builtin_fabsf(v));
        nothing = __builtin_fmaf(y, 0.0f, nothing);
        sums[i][j][r] = y;
      }
  }
  return {nothing != 0.0f, least < SAFE_SUM};
}
// Could a sum (unscaled by now) show what was lost?  lossy: how many elements of each of the wavefront's columns lose bits (each
// = 1), or of all of them together (0).
template <bool PACKED_ROWS, int QB>
__device__ __forceinline__ bool shows_loss(const HalfSums<QB> &sums, const HalfOperand &w, const unsigned *lossy, int each, int strip0, int np, int q0,
                                           int nq, int eq, int depth) {
  const int *const exps = reinterpret_cast<const int *>(w.packed + half_fragment_bytes(w.strips, w.steps));
  const unsigned *const words = reinterpret_cast<const unsigned *>(exps + w.strips * 16);
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  bool shows = false;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    unsigned theirs = 0;
    for (int c = 0; strip0 + i < w.strips && c < w.chunks; c++) theirs += words[(strip0 + i) * w.chunks + c];
#pragma unroll
    for (int j = 0; j < QB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = (strip0 + i) * 16 + (PACKED_ROWS ? 4 * g4 + r : c16), q = 16 * j + (PACKED_ROWS ? c16 : 4 * g4 + r);
        const unsigned count = theirs + lossy[each * q];
        const float v = __builtin_ldexpf(sums[i][j][r], exps[row < np ? row : 0] + eq);
        shows |= count && row < np && q0 + q < nq && __builtin_fabsf(v) * (float)depth < SAFE_SUM * (float)count;
      }
  }
  return shows;
}
// Blocks of 16 x 16 -> blocks of 32 x 32 as v_mfma_f32_32x32x2_f32 leaves them.
template <bool PACKED_ROWS, int QB, int MT, int NT>
__device__ __forceinline__ void to_blocks(const HalfSums<QB> &sums, f32x16 (&acc)[MT][NT]) {
#pragma unroll
  for (int R = 0; R < MT; R++)
#pragma unroll
    for (int C = 0; C < NT; C++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          float a = PACKED_ROWS ? sums[i][2 * C][r] : sums[0][2 * R + i][r];
          float b = PACKED_ROWS ? sums[i][2 * C + 1][r] : sums[1][2 * R + i][r];
          swap16(a, b);
          swap32(a, b);
          acc[R][C][8 * i + r] = a;
          acc[R][C][8 * i + 4 + r] = b;
        }
}
// The sums of KG groups of THREADS each, in order; those behind the first leave theirs in LDS, `stride` bytes apart.  False: not
// the group that goes on.
template <int KG, int THREADS, int MT, int NT>
__device__ __forceinline__ bool join_groups(f32x16 (&acc)[MT][NT], unsigned char *base, int stride, int group, int tid) {
  if (group > 0) {
    float *const mine = reinterpret_cast<float *>(base + (group - 1) * stride);
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < NT; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) mine[((a * NT + b) * 16 + r) * THREADS + tid] = acc[a][b][r];
  }
  __syncthreads();
  if (group > 0) return false;
#pragma unroll
  for (int g = 1; g < KG; g++) {
    const float *const other = reinterpret_cast<const float *>(base + (g - 1) * stride);
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < NT; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] += other[((a * NT + b) * 16 + r) * THREADS + tid];
  }
  return true;
}
// The largest magnitude (as bits) that the threads of a group have met; `most`: a word for each of its WAVES wavefronts.
template <int WAVES>
__device__ __forceinline__ unsigned group_most(unsigned top, unsigned *most, int wave) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const unsigned u = __shfl_xor(top, d);
    top = u > top ? u : top;
  }
  if ((threadIdx.x & 63) == 0) most[wave] = top;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < WAVES; i++) top = most[i] > top ? most[i] : top;
  return top;
}

// WP wavefronts of 32 packed rows x BQ columns of the other operand; KG groups of them share K.
template <int WP, int BQ, int KG, int SRC>
__global__ __launch_bounds__(WP * KG * 64, 2) void half_kernel(Params p, HalfOperand w) {
  constexpr bool CONV = SRC == H_PIXELS;
  constexpr int THREADS = WP * 64, BP = WP * 32, QB = BQ / 16;
  constexpr int BM = CONV ? BP : BQ, BN = CONV ? BQ : BP, WM = CONV ? WP : 1, WN = CONV ? 1 : WP;
  constexpr int PLANE = BQ * 16, BUF = 16 * PLANE;
  __shared__ __attribute__((aligned(16))) unsigned char lds_all[KG][2][BUF];
  __shared__ unsigned most[KG * WP];
  static_assert(2 * BUF >= WM * WN * STAGE_FLOATS * 4, "epilogue staging");
  static_assert(KG == 1 || 2 * BUF >= BM * BN * 4, "partial sums");

  const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);
  unsigned char(*const lds)[BUF] = lds_all[group];
  const int tid = (int)threadIdx.x - group * THREADS;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g4 = lane >> 4;

  const TileWork tw = decode_work(p, (int)blockIdx.x);
  const int row0 = tw.tm * BM, col0 = tw.tn * BN;
  const int p0 = CONV ? row0 : col0, q0 = CONV ? col0 : row0;  // first packed row, first column of the other operand
  const int np = CONV ? p.m : p.n, nq = CONV ? p.n : p.m;
  const int kfirst = tw.whole ? 0 : tw.chunk * p.kchunk;
  const int klast = tw.whole ? p.k : (kfirst + p.kchunk < p.k ? kfirst + p.kchunk : p.k);
  const int kshare = ((klast - kfirst + HK - 1) / HK + KG - 1) / KG * HK;
  const int kbeg = kfirst + group * kshare, kend = kbeg + kshare < klast ? kbeg + kshare : klast;
  const int blocks = kshare / HK;

  // ---- the other operand: eight k of a column at a time ---------------------------------------------------
  constexpr int G8 = THREADS / BQ;                                 // pixels: a wavefront has one of the G8 eights
  constexpr int NJ = 8 * BQ / THREADS;
  const int ld = (int)(CONV ? p.sB0 : p.sA0);
  auto pixel = [&](int col) -> int {
    const unsigned P = (unsigned)col < (unsigned)p.n ? (unsigned)col : (unsigned)p.n - 1;
    const unsigned plane = (unsigned)(p.cv.h * p.cv.w), ohw = (unsigned)(p.cv.oh * p.cv.ow);
    const unsigned img = (unsigned)fdiv((int)P, p.cv.fd_ohw), q = P - img * ohw;
    const unsigned oy = (unsigned)fdiv((int)q, p.cv.fd_ow), ox = q - oy * (unsigned)p.cv.ow;
    return (int)(img * (unsigned)p.cv.c_total * plane) + (int)oy * p.cv.sh * p.cv.w + (int)ox * p.cv.sw;
  };
  const int k8 = CONV ? __builtin_amdgcn_readfirstlane(tid / BQ) : tid & 7;
  const int qcol = CONV ? tid % BQ : tid >> 3;
  int voff[CONV ? 1 : NJ];
  if (CONV) {
    voff[0] = pixel(q0 + qcol) * 4;
  } else {
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      int r = q0 + qcol + j * (THREADS / 8);
      r = r < nq ? r : nq - 1;  // rows past the last repeat it: their sums are never stored
      voff[CONV ? 0 : j] = (r * ld + k8 * 8) * 4;
    }
  }
  const rsrc_t rsrc_q = make_rsrc(CONV ? p.B : p.A, CONV ? p.b_bytes : p.a_bytes);
  struct Eights { float x[NJ][8]; } next;
  auto fetch_eight = [&](int k0, Eights &s, int j) {
    if constexpr (CONV) {
      const int k = k0 + 8 * (k8 + G8 * j);
      const int v = k < kend ? voff[0] : BUF_OOB;  // (k % 8 == 0)
#pragma unroll
      for (int e = 0; e < 8; e++) s.x[j][e] = buf_load(rsrc_q, v, (k + e) * ld * 4);
    } else {
      const int v = k0 + 8 * k8 < kend ? voff[CONV ? 0 : j] : BUF_OOB;
      const f32x4 a = buf_load4(rsrc_q, v, k0 * 4), b = buf_load4(rsrc_q, v, k0 * 4 + 16);
#pragma unroll
      for (int e = 0; e < 4; e++) s.x[j][e] = a[e], s.x[j][4 + e] = b[e];
    }
  };
  auto fetch = [&](int k0, Eights &s) {
#pragma unroll
    for (int j = 0; j < NJ; j++) fetch_eight(k0, s, j);
  };
  float sq = 1.0f;
  int eq = 0;
  auto put = [&](unsigned char *buf, const Eights &s, int j) {
    const HalfParts q = half_parts(s.x[j], sq);
    const int plane = CONV ? k8 + G8 * j : k8, col = CONV ? qcol : qcol + j * (THREADS / 8);
    unsigned char *const cell = buf + plane * PLANE + (col ^ 2 * plane) * 16;
    *reinterpret_cast<f16x8 *>(cell) = q.h;
    *reinterpret_cast<f16x8 *>(cell + 8 * PLANE) = q.l;
  };

  // ---- the packed operand: from L2 straight into the lanes -------------------------------------------------
  const rsrc_t rsrc_p = make_rsrc(w.packed, (int)half_fragment_bytes(w.strips, w.steps));
  const int strip0 = p0 / 16 + wave * 2, stripsize = w.steps * STEP_BYTES;
  struct Strips { f16x8 h[2][2], l[2][2]; } strips[2];  // [strip][32 k]
  auto fetch_strips = [&](int k0, Strips &s) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // (past the last strip, or the last step: some other one again, whose sums are never stored.  A scalar offset is no part of what
      // a descriptor is checked for, so it stays within the block.)
      const int strip = strip0 + i < w.strips ? strip0 + i : w.strips - 1, step = k0 / HSTEP < w.steps ? k0 / HSTEP : 0;
      const int soff = strip * stripsize + step * STEP_BYTES;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        s.h[i][t] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, lane * 16, soff + t * STEP_BYTES, 0));
        s.l[i][t] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, lane * 16 + 1024, soff + t * STEP_BYTES, 0));
      }
    }
  };

  f32x4 total[2][QB];  // [strip][16 columns]
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < QB; j++) total[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto mul = [](f16x8 a, f16x8 b, f32x4 c) {
    return CONV ? __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a, c, 0, 0, 0);
  };

  // the first block says what the others are scaled by
  fetch(kbeg, next);
  fetch_strips(kbeg, strips[0]);
  unsigned top = 0;
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const unsigned u = __float_as_uint(next.x[j][e]) & 0x7fffffffu;
      top = u > top ? u : top;
    }
  top = group_most<WP>(top, most + group * WP, wave);
  eq = __builtin_amdgcn_readfirstlane(scale_exponent(top, X_TARGET));
  sq = scale_of(eq);
#pragma unroll
  for (int j = 0; j < NJ; j++) put(lds[0], next, j);
  fetch(kbeg + HK, next);
  __syncthreads();

  // A group: two strips x 16 columns.  Its fragments are read under the products of the group before it, its sums added to the
  // totals under those of the group behind it; the barrier of a block stands before its last group, whose products are
  // under the reads of the next block's first.
  struct Columns { f16x8 h[2], l[2]; } columns[2];  // [32 k]
  auto read_columns = [&](int cur, int j, Columns &c) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const unsigned char *const at = lds[cur] + (4 * t + g4) * PLANE + (c16 ^ (2 * g4 + 8 * t)) * 16 + j * 256;
      c.h[t] = *reinterpret_cast<const f16x8 *>(at);
      c.l[t] = *reinterpret_cast<const f16x8 *>(at + 8 * PLANE);
    }
  };
  f32x4 high[2], low[2];
#pragma unroll
  for (int i = 0; i < 2; i++) high[i] = low[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto flush = [&](int j) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
      for (int r = 0; r < 4; r++) total[i][j][r] += __builtin_fmaf(low[i][r], 1.0f / LOW_SCALE, high[i][r]);
      asm volatile("" : "+v"(total[i][j]));
    }
  };
  read_columns(0, 0, columns[0]);
  auto block = [&](int k0, int cur) {
    const Strips &s = strips[cur];
    fetch_strips(k0 + HK, strips[cur ^ 1]);
#pragma unroll
    for (int j = 0; j < QB; j++) {
      const Columns &c = columns[j & 1];
      if (j + 1 < QB) {
        read_columns(cur, j + 1, columns[(j + 1) & 1]);
      } else {
        __syncthreads();
        read_columns(cur ^ 1, 0, columns[0]);
      }
      f32x4 h[2], l[2];
      auto products = [&](const f16x8 (&a)[2][2], int t, f16x8 b, f32x4 (&sum)[2], bool first) {
#pragma unroll
        for (int i = 0; i < 2; i++) sum[i] = mul(a[i][t], b, first ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : sum[i]);
      };
      products(s.h, 0, c.l[0], l, true);
      products(s.h, 0, c.h[0], h, true);
      products(s.l, 0, c.h[0], l, false);
      products(s.h, 1, c.h[1], h, false);
      products(s.h, 1, c.l[1], l, false);
      products(s.l, 1, c.h[1], l, false);
      flush((j + QB - 1) % QB);
      // the next block goes to the other buffer between the products, and the one behind it is requested
      constexpr int EVERY = (QB - 2) / NJ > 0 ? (QB - 2) / NJ : 1;
      const bool puts = j % EVERY == 0 && j / EVERY < NJ;
      if (puts) {
        put(lds[cur ^ 1], next, j / EVERY);
        fetch_eight(k0 + 2 * HK, next, j / EVERY);
      }
#pragma unroll
      for (int i = 0; i < 2; i++) high[i] = h[i], low[i] = l[i];
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 12; i++) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        if (puts) __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        else __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int b = 0;
  for (; b + 1 < blocks; b += 2) {
    block(kbeg + b * HK, 0);
    block(kbeg + b * HK + HK, 1);
  }
  if (b < blocks) block(kbeg + b * HK, 0);
  flush(QB - 1);

  // ---- unscaled; is there anything the two parts could not hold? ------------------------------------------
  const HalfDoubt doubt = unscale<CONV, QB>(total, w, strip0, np, eq);
  bool again = false;
  if (__syncthreads_or(doubt.bad || doubt.tiny)) {
    again = __syncthreads_or(doubt.bad);
    if (!again) {
      // (which columns hold such elements, and how many?)
      unsigned *const lossy = reinterpret_cast<unsigned *>(&lds[0][0]);
      for (int i = tid; i < BQ; i += THREADS) lossy[i] = 0;
      __syncthreads();
      const float least = __builtin_ldexpf(1.0f, FULL_EXPONENT - eq);
      for (int k0 = kbeg; k0 < kend; k0 += HK) {
        fetch(k0, next);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          unsigned count = 0;
#pragma unroll
          for (int e = 0; e < 8; e++) count += __builtin_fabsf(next.x[j][e]) < least && next.x[j][e] != 0.0f ? 1u : 0u;
          if (count) atomicAdd(&lossy[CONV ? qcol : qcol + j * (THREADS / 8)], count);
        }
      }
      __syncthreads();
      again = __syncthreads_or(kend > kbeg && shows_loss<CONV, QB>(total, w, lossy, 1, strip0, np, q0, nq, eq, kend - kbeg));
    }
  }
  constexpr int MT = CONV ? 1 : BQ / 32, NT = CONV ? BQ / 32 : 1;
  f32x16 acc[MT][NT];
  to_blocks<CONV, QB>(total, acc);
  if (KG > 1 && !again && !join_groups<KG, THREADS>(acc, &lds_all[0][0][0], 2 * BUF, group, tid)) return;
  if (again) {
    if (KG > 1) __syncthreads();
    if (group > 0) return;
    // the fp32 instruction, operands as they lie: [row or column][16 k, 4 apart]
    constexpr int LDW = BK + 4;
    static_assert((BM + BN) * LDW * 4 <= 2 * BUF, "whole slabs");
    float *const raw = reinterpret_cast<float *>(&lds[0][0]);
    const int li = lane & 31, half = lane >> 5;
    const bool p_kc = CONV || p.sB0 == 1;
    const float *const praw = CONV ? p.A : p.B;
    const long long ps = CONV ? p.sA0 : p.sB1, pk = CONV ? 1 : p.sB0;
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < NT; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
    float *const fp = raw + (CONV ? 0 : BM * LDW), *const fo = raw + (CONV ? BM * LDW : 0);
    constexpr int PP = BP * BK / THREADS, PQ = BQ * BK / THREADS;
    float a[PP], b[PQ];
    auto fetch_whole = [&](int k0) {
#pragma unroll
      for (int i = 0; i < PP; i++) {
        const int id = tid + i * THREADS, r = p_kc ? id / BK : id % BP, k = k0 + (p_kc ? id % BK : id / BP);
        a[i] = p0 + r < np && k < klast ? praw[(p0 + r) * ps + k * pk] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < PQ; i++) {
        const int id = tid + i * THREADS, r = CONV ? id % BQ : id / BK, k = k0 + (CONV ? id / BQ : id % BK);
        const int at = k < klast ? k : 0, v = (CONV ? voff[0] / 4 + at * ld : (q0 + r < nq ? q0 + r : nq - 1) * ld + at) * 4;
        b[i] = buf_load(rsrc_q, k < klast ? v : BUF_OOB, 0);
      }
    };
    fetch_whole(kfirst);
    for (int k0 = kfirst; k0 < klast; k0 += BK) {
      __syncthreads();  // everybody has read the slab before
#pragma unroll
      for (int i = 0; i < PP; i++) {
        const int id = tid + i * THREADS, r = p_kc ? id / BK : id % BP, k = p_kc ? id % BK : id / BP;
        fp[r * LDW + k] = a[i];
      }
#pragma unroll
      for (int i = 0; i < PQ; i++) {
        const int id = tid + i * THREADS, r = CONV ? id % BQ : id / BK, k = CONV ? id / BQ : id % BK;
        fo[r * LDW + k] = b[i];
      }
      __syncthreads();
      fetch_whole(k0 + BK);
      const float *const fa = raw + ((CONV ? wave * 32 : 0) + li) * LDW + 8 * half, *const fb = raw + (BM + (CONV ? 0 : wave * 32) + li) * LDW + 8 * half;
      f32x4 ea[MT][2], eb[NT][2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int t = 0; t < MT; t++) ea[t][h] = *reinterpret_cast<const f32x4 *>(fa + t * 32 * LDW + 4 * h);
#pragma unroll
        for (int t = 0; t < NT; t++) eb[t][h] = *reinterpret_cast<const f32x4 *>(fb + t * 32 * LDW + 4 * h);
      }
#pragma unroll
      for (int e = 0; e < 8; e++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int nt = 0; nt < NT; nt++)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ea[mt][e >> 2][e & 3], eb[nt][e >> 2][e & 3], acc[mt][nt], 0, 0, 0);
    }
    __syncthreads();
  }
  finish_tile<BM, BN, WM, WN, CONV, 2>(p, acc, tw.whole, tw.lin, tw.chunk, 0, row0, col0, reinterpret_cast<float *>(&lds[0][0]) + wave * STAGE_FLOATS);
}

template <int WP, int BQ, int KG, int SRC>
int launch_half_tile(Params &p, const HalfOperand &w, const WorkPlan &work) {
  constexpr int BP = WP * 32;
  return launch_planned<SRC == H_PIXELS ? BP : BQ, SRC == H_PIXELS ? BQ : BP>(p, 1, SRC == H_PIXELS, HK, 0, [&](dim3 grid, bool) {
    hipLaunchKernelGGL((half_kernel<WP, BQ, KG, SRC>), grid, dim3(WP * KG * 64), 0, wdh::stream(), p, w);
  }, &work);
}
template <int SRC>
int launch_half(const HalfPlan &s, Params &p, const HalfOperand &w) {
  switch (s.tile) {
    case H256x128: return launch_half_tile<8, 128, 1, SRC>(p, w, s.work);
    case H128x128: return launch_half_tile<4, 128, 1, SRC>(p, w, s.work);
    case H128x64: return launch_half_tile<4, 64, 1, SRC>(p, w, s.work);
    default: return launch_half_tile<4, 64, 2, SRC>(p, w, s.work);
  }
}

}  // namespace wdhc

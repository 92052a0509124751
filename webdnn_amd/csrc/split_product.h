// Products of fp32 operands on the bf16 matrix cores, without giving up fp32 accuracy.
//
// A float is the exact sum of three bfloat16 values: h = x rounded to the nearest one, m = x - h rounded likewise, and
// l = x - h - m (both subtractions are exact, and what is left fits eight bits).  Of the nine products of two such sums
// the three below 2^-25 of the whole (m*l, l*m, l*l) are left out; the other six go through
// v_mfma_f32_32x32x16_bf16, which multiplies sixteen times as many pairs a cycle as v_mfma_f32_32x32x2_f32 and adds in
// fp32.  Rounding to nearest matters: with the upper sixteen bits instead the parts share a sign, what is left out too, and
// every product is 3e-8 too small, which fifty layers add up (ResNet-50's logits 2.4e-3 off where 1e-3 is allowed; 6e-4 now).
// The matrix core adds a product to a far larger sum less exactly than a fused multiply-add does, so the leading
// products h*h and the five small ones are summed apart and meet once at the end: a chain has K/16 (small ones:
// 5K/16) additions where the fp32 instruction makes K/2.  Errors against 64 bits (2-norm, normally distributed operands, fp32
// instruction / this): K 64 14.5e-8 / 5.0e-8, 256 28.7e-8 / 8.9e-8, 1024 5.8e-7 / 1.9e-7, 4096 11.5e-7 / 4.0e-7; positive
// operands 12.2e-8 / 5.2e-8 to 9.8e-7 / 3.5e-7, no drift to either side (below 1e-8).
//
// Bound: power, then instruction issue.  A loop of nothing but these instructions on normally distributed operands runs at 1720 to
// 1770 TFLOP/s and 1.8 GHz (on zeros 2320 and 2.4), which is 290 of fp32 products (the fp32 instruction's own limit is 157); at
// 4096^3 the clock is the same and the matrix cores are busy 70 % of the cycles (counters in
// profiles/contraction_kernel_gemm4096_conv_c3.txt).  What a slab adds to the products is the split (14 vector instructions per pair of elements, three of
// them to look at it) and LDS traffic (6 bytes an element), so an operand is split once, on its way from registers to LDS,
// not by every wavefront that multiplies it.  The split and the LDS stores of the next slab are placed between the matrix
// instructions of this one (sched_group_barrier): 195 -> 209 TFLOP/s, because the wavefronts of a SIMD else meet the same phase
// at the same time.  Measured at 4096^3 (TFLOP/s; fp32 instruction 146): 64x64 tiles 159, 64x128 and 128x64 181, 128x128 209,
// 256x128 210 to 222.  Tried without gain: fragments of the next slab read ahead (204), loads two to eight slabs ahead (204), small
// products in two or three chains; LDS planes without the 64 bytes between their halves (a third more LDS cycles, 198).
//
// What the split cannot hold is done again with the fp32 instruction, a whole tile (or chunk) at a time:
//   * an Inf or NaN operand leaves NaN in x - h and therefore in every sum it enters; so does a sum that overflows;
//   * bfloat16 ends at 2^-133 (parts and results below 2^-126 are kept, by the conversion and by the matrix instruction): an element
//     below 2^-110 loses up to 2^-134, one below 2^-134 all of itself.  So every element is looked at where it is split (least_of).
//     The sums cannot tell: large partners lift what is left of such an element to any size, and one that vanished leaves a
//     zero.  A tile with such elements is done again unless all its sums are at least 2^-60 and no operand element reaches
//     2^30: then K terms are off by at most K 2^-104, beyond the last bits of the sums.  (That keeps softmax rows and
//     weights with a few vanishing elements on the fast path.  The look costs ResNet-50 of 128 images 6986 -> 7045 us, products in
//     256x128 tiles nothing (see BY_PAIR).)
#pragma once
#include "contraction.h"

namespace wdhc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// Two elements -> their three parts, packed (the first in the lower sixteen bits).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
struct SplitPair { unsigned h, m, l; float r0, r1; };  // r: what l is the nearest value to
__device__ __forceinline__ unsigned nearest_pair(float x0, float x1) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
}
__device__ __forceinline__ SplitPair split_pair(float x0, float x1) {
  const unsigned h = nearest_pair(x0, x1);
  const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  const unsigned m = nearest_pair(r0, r1);
  const float s0 = r0 - __uint_as_float(m << 16), s1 = r1 - __uint_as_float(m & 0xffff0000u);
  return SplitPair{h, m, nearest_pair(s0, s1), s0, s1};
}

// The least nonzero magnitude of what was split, as doubled bits less one (a zero becomes the largest), and what it and the sums say.
__device__ __forceinline__ unsigned least_of(unsigned least, float x0, float x1) {
  const unsigned u0 = (__float_as_uint(x0) << 1) - 1u, u1 = (__float_as_uint(x1) << 1) - 1u;
  const unsigned u = u0 < u1 ? u0 : u1;
  return u < least ? u : least;
}
constexpr unsigned doubled_bits(int exponent) { return (unsigned)(127 + exponent) << 24; }
__device__ __forceinline__ bool loses_bits(unsigned least) { return least < doubled_bits(-110) - 1u; }
// The same asked of a pair by itself: only what is left of small elements (below 2^-102) is subnormal and not zero.
__device__ __forceinline__ bool may_lose_bits(const SplitPair &s) {
  constexpr int SUBNORMAL = 0x90;  // (of either sign)
  return __builtin_amdgcn_classf(s.r0, SUBNORMAL) | __builtin_amdgcn_classf(s.r1, SUBNORMAL);
}
__device__ __forceinline__ bool reaches_partners(float x) { return (__float_as_uint(x) << 1) >= doubled_bits(30); }
__device__ __forceinline__ bool reaches_partners(f32x4 v) {
  return reaches_partners(v.x) | reaches_partners(v.y) | reaches_partners(v.z) | reaches_partners(v.w);
}
// The range of a tile's sums, as doubled bits.
struct SumRange { unsigned least, most; };
__device__ __forceinline__ void add_sum(SumRange &g, float x) {
  const unsigned u = __float_as_uint(x) << 1;
  g.most = u > g.most ? u : g.most;
  g.least = u < g.least ? u : g.least;
}
__device__ __forceinline__ bool not_finite(const SumRange &g) { return g.most >= doubled_bits(128); }
__device__ __forceinline__ bool small_sums(const SumRange &g) { return g.least < doubled_bits(-60); }

// Workgroups a CU holds: the accumulators are two per result, so 128x128 tiles take 64 + 64 registers of
// accumulators and two of them fit; 256x128 is the same wavefront with eight of them in one workgroup.
constexpr int split_blocks(int bm, int bn) { return bm * bn >= 128 * 128 ? 2 : (bm * bn > 64 * 64 ? 3 : 4); }

// LDS: three planes (h, m, l) per operand, each [k / 8][row or column][8 bf16], so that a fragment of a 32x16 block
// is one 16-byte read per lane, 32 lanes side by side.
//
// KG: groups of WM x WN wavefronts that share the K of a tile, each with LDS of its own; their sums meet in LDS, in
// order.  A 64x64 tile by itself on a CU keeps one wavefront a SIMD, which issues its 110 instructions a slab one after
// the other in 0.29 us, where the products alone take 0.08; two groups take 0.20 for a slab, four 0.16.  (us, one / two / four:
// 384x2304x768 21.2 / 18.0 / 16.8, 1024^3 26.8 / 22.6 / 21.3, 8 images 512 -> 512 on 14x14 16.6 / 14.3 / 13.8; with two tiles a CU
// there is nothing to gain, 850x2048x256 13.3 / 13.2 / 18.2.)
template <int BM, int BN, int WM, int WN, int BMODE, int KG>
__device__ __forceinline__ void split_tile(const Params &p, int pid) {
  constexpr int THREADS = WM * WN * 64;  // of a group
  constexpr bool IM2COL = BMODE == B_IM2COL32 || BMODE == B_IM2COL64;
  constexpr bool PIX_ANY = BMODE == B_PIXELS_ANY;
  constexpr bool PIXELS = BMODE == B_PIXELS || PIX_ANY;
  constexpr bool CONV = IM2COL || PIXELS;
  constexpr bool B_IS_KC = BMODE == B_KC;
  constexpr bool B_COLUMNS = !B_IS_KC && !IM2COL;  // B contiguous along its columns
  constexpr int MT = BM / (WM * 32), NT = BN / (WN * 32);
  // (bytes; the 64 between the halves of a plane keep the 8-byte stores of 16 lanes, four k of each of eight rows, on
  // different banks)
  constexpr int HALF_A = BM * 16 + 64, HALF_B = BN * 16 + 64, PLANE_A = 2 * HALF_A, PLANE_B = 2 * HALF_B;
  constexpr int BUF = 3 * (PLANE_A + PLANE_B);
  __shared__ __attribute__((aligned(16))) unsigned char lds_all[KG][2][BUF];
  static_assert(2 * BUF >= WM * WN * STAGE_FLOATS * 4, "epilogue staging");
  static_assert(KG == 1 || 2 * BUF >= BM * BN * 4, "partial sums");

  const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);
  unsigned char(*const lds)[BUF] = lds_all[group];
  const int tid = (int)threadIdx.x - group * THREADS;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 31, half = lane >> 5;
  const int wrow = wm * (MT * 32), wcol = wn * (NT * 32);

  const TileWork tw = decode_work(p, pid);
  const int bz = tw.bz, row0 = tw.tm * BM, col0 = tw.tn * BN;
  const int kfirst = tw.whole ? 0 : tw.chunk * p.kchunk;
  const int klast = tw.whole ? p.k : (kfirst + p.kchunk < p.k ? kfirst + p.kchunk : p.k);
  const int kshare = KG == 1 ? klast - kfirst : ((klast - kfirst + BK - 1) / BK + KG - 1) / KG * BK;
  const int kbeg = kfirst + group * kshare;   // (a group may have less than the others, or nothing: zeros, then)
  int kend = KG == 1 || kbeg + kshare < klast ? kbeg + kshare : klast;
  const float *const A = p.A + (long long)bz * p.sAb;
  const float *const B = CONV ? p.B + (long long)bz * p.cv.c_in_g * p.cv.h * p.cv.w : p.B + (long long)bz * p.sBb;
  const int lda = (int)p.sA0, ldb = (int)(B_IS_KC ? p.sB1 : p.sB0);

  // ---- fetch plans: one byte offset per piece, every address term folded in -------------------------
  // k-contiguous: thread t takes k 4*(t%4)..+3 of rows t/4 + i*THREADS/4.
  constexpr int RPP = THREADS / 4, NA = BM / RPP;
  static_assert(NA >= 1 && BM % RPP == 0, "rows per pass");
  const int kq = tid & 3;
  int voff_a[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    int r = row0 + (tid >> 2) + i * RPP;
    r = r < p.m ? r : p.m - 1;  // rows and columns past the edge feed only sums that are never stored
    voff_a[i] = (r * lda + kq * 4) * 4;
  }
  const rsrc_t rsrc_a = make_rsrc(A, p.a_bytes);

  // column-contiguous: a piece is four k of CPP neighbouring columns.  Neighbouring lanes take the lower and the
  // upper four k of one plane row, so that their 8-byte LDS stores lie side by side.
  constexpr int CPP = BN * 4 / THREADS;  // columns per thread (1 or 2)
  constexpr int NB = B_IS_KC ? BN / RPP : 1;
  constexpr int G = THREADS / BN > 0 ? THREADS / BN : 1, L = BK / G;  // im2col: L consecutive k of one pixel
  static_assert(!B_COLUMNS || CPP == 1 || CPP == 2, "column pieces");
  static_assert(!IM2COL || (L == 4 || L == 8), "im2col pieces");
  const int bkq = B_COLUMNS ? (tid & 1) | ((tid / (2 * (BN / CPP))) << 1) : 0;
  const int bcol = B_COLUMNS ? ((tid >> 1) % (BN / CPP)) * CPP : 0;
  int voff_b[B_IS_KC ? NB : CPP];
  PixelFast pf = {0, 0xffffffffu, 0xffffffffu};
  const int bias = IM2COL ? p.cv.pt * p.cv.w + p.cv.pl : 0;  // makes every corner offset >= 0
  const int kgroup0 = IM2COL ? __builtin_amdgcn_readfirstlane(tid / BN) * L : 0;
  // element offset of a column of B at k = 0 (conv: of a pixel of the group's first channel; im2col: of the
  // receptive field's corner, plus `bias`)
  auto column = [&](int col) -> int {
    if (!CONV) return col;
    // (columns past the last repeat it, or the last pair where they are read in pairs)
    constexpr unsigned LAST = BMODE == B_PIXELS ? CPP : 1;
    const unsigned P = (unsigned)col < (unsigned)p.n ? (unsigned)col : (unsigned)p.n - LAST;
    const unsigned plane = (unsigned)(p.cv.h * p.cv.w), ohw = (unsigned)(p.cv.oh * p.cv.ow);
    const unsigned img = (unsigned)fdiv((int)P, p.cv.fd_ohw), q = P - img * ohw;
    const unsigned oy = (unsigned)fdiv((int)q, p.cv.fd_ow), ox = q - oy * (unsigned)p.cv.ow;
    return (int)(img * (unsigned)p.cv.c_total * plane) + ((int)oy * p.cv.sh - (IM2COL ? p.cv.pt : 0)) * p.cv.w +
           (int)ox * p.cv.sw - (IM2COL ? p.cv.pl : 0) + bias;
  };
  auto padding = [&](int col, PixelFast &f) {  // which taps of this pixel lie in the padding
    f.pad_lo = f.pad_hi = 0xffffffffu;
    if (col >= p.n) return;
    const unsigned ohw = (unsigned)(p.cv.oh * p.cv.ow);
    const unsigned q = (unsigned)col - (unsigned)fdiv(col, p.cv.fd_ohw) * ohw;
    const int oy = fdiv((int)q, p.cv.fd_ow), ox = (int)q - oy * p.cv.ow;
    unsigned long long inside = 0;
    int t = 0;
    for (int ky = 0; ky < p.cv.kh; ky++) {
      const bool row_in = (unsigned)(oy * p.cv.sh - p.cv.pt + ky * p.cv.dh) < (unsigned)p.cv.h;
      for (int kx = 0; kx < p.cv.kw; kx++, t++)
        if (row_in && (unsigned)(ox * p.cv.sw - p.cv.pl + kx * p.cv.dw) < (unsigned)p.cv.w) inside |= 1ull << t;
    }
    f.pad_lo = ~(unsigned)inside;
    f.pad_hi = ~(unsigned)(inside >> 32);
  };
  if (B_IS_KC) {
#pragma unroll
    for (int i = 0; i < NB; i++) {
      int c = col0 + (tid >> 2) + i * RPP;
      c = c < p.n ? c : p.n - 1;
      voff_b[i] = (c * ldb + kq * 4) * 4;
    }
  } else if (IM2COL) {
    const int col = col0 + tid % BN;
    pf.valid = column(col) * 4;
    padding(col, pf);
  } else {
#pragma unroll
    for (int i = 0; i < CPP; i++)  // (columns past a matrix may hold anything: they read as zeros)
      voff_b[i] = CONV || col0 + bcol + i < p.n ? (bkq * 4 * ldb + column(col0 + bcol + i)) * 4 : BUF_OOB;
  }
  const int b_window = CONV ? p.b_bytes - (int)((long long)bz * p.cv.c_in_g * p.cv.h * p.cv.w * 4) : p.b_bytes;
  const rsrc_t rsrc_b = make_rsrc(B - bias, b_window);

  struct Slab {
    f32x4 a[NA];
    f32x4 b[B_IS_KC ? NB : (IM2COL ? L / 4 : CPP)];  // four consecutive k each
  };
  // im2col: the tap table's entries of the slab to be fetched next (scalar loads, a slab ahead of their use)
  struct { int2 e[IM2COL ? L : 1]; } taps;
  const int ktab_last = IM2COL ? (p.k + BK - 1) / BK * BK - BK : 0;
  auto read_taps = [&](int k0) {
    if (!IM2COL) return;
    k0 = k0 < ktab_last ? k0 : ktab_last;
#pragma unroll
    for (int i = 0; i < (IM2COL ? L : 1); i++) taps.e[i] = p.cv.ktab[k0 + kgroup0 + i];
  };
  // last: the slab may reach past kend (a multiple of four): pieces beyond it read as zeros
  auto fetch = [&](int k0, Slab &s, bool last) {
#pragma unroll
    for (int i = 0; i < NA; i++)
      s.a[i] = buf_load4(rsrc_a, last && k0 + kq * 4 >= kend ? BUF_OOB : voff_a[i], k0 * 4);
    if (B_IS_KC) {
#pragma unroll
      for (int i = 0; i < NB; i++)
        s.b[i] = buf_load4(rsrc_b, last && k0 + kq * 4 >= kend ? BUF_OOB : voff_b[i], k0 * 4);
    } else if (IM2COL) {
#pragma unroll
      for (int i = 0; i < L; i++) {
        const int2 e = taps.e[i];
        const unsigned word = (BMODE == B_IM2COL64 && (e.y & 32)) ? pf.pad_hi : pf.pad_lo;
        const int pad = __builtin_amdgcn_sbfe((int)word, (unsigned)e.y & 31u, 1u);
        s.b[i >> 2][i & 3] = buf_load(rsrc_b, (pad & BUF_OOB) | pf.valid, e.x);
      }
      read_taps(k0 + BK);
    } else {
      const bool out = last && k0 + bkq * 4 >= kend;
      const int voff = out ? BUF_OOB : voff_b[0];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int soff = (k0 + e) * ldb * 4;
        if (CPP == 1) {
          s.b[0][e] = buf_load(rsrc_b, voff, soff);
        } else if (PIX_ANY) {
          s.b[0][e] = buf_load(rsrc_b, voff, soff);
          s.b[CPP - 1][e] = buf_load(rsrc_b, out ? BUF_OOB : voff_b[CPP - 1], soff);
        } else {
          const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc_b, voff, soff, 0));
          s.b[0][e] = v.x;
          s.b[CPP - 1][e] = v.y;
        }
      }
    }
  };
  // Were there elements that lose bits?  The least of them takes three vector instructions a pair, each by itself two and two
  // scalar ones, which wide tiles have the slots for (us, 4096^3 with 256x128 tiles 652 / 634, without either 638; 384x3072x768
  // 26.6 / 27.5, 26.5).
  constexpr bool BY_PAIR = BM * BN > 128 * 128;
  unsigned least = 0xffffffffu;
  bool lost = false;
  auto put4 = [&](unsigned char *cell, int plane, f32x4 v) {
    const SplitPair lo = split_pair(v.x, v.y), hi = split_pair(v.z, v.w);
    if (BY_PAIR) lost = lost | may_lose_bits(lo) | may_lose_bits(hi);
    else least = least_of(least_of(least, v.x, v.y), v.z, v.w);
    *reinterpret_cast<u32x2 *>(cell) = u32x2{lo.h, hi.h};
    *reinterpret_cast<u32x2 *>(cell + plane) = u32x2{lo.m, hi.m};
    *reinterpret_cast<u32x2 *>(cell + 2 * plane) = u32x2{lo.l, hi.l};
  };
  auto put = [&](unsigned char *buf, const Slab &s) {
    unsigned char *const b = buf + 3 * PLANE_A;
#pragma unroll
    for (int i = 0; i < NA; i++)
      put4(buf + (kq >> 1) * HALF_A + ((tid >> 2) + i * RPP) * 16 + (kq & 1) * 8, PLANE_A, s.a[i]);
    if (B_IS_KC) {
#pragma unroll
      for (int i = 0; i < NB; i++)
        put4(b + (kq >> 1) * HALF_B + ((tid >> 2) + i * RPP) * 16 + (kq & 1) * 8, PLANE_B, s.b[i]);
    } else if (IM2COL) {
#pragma unroll
      for (int i = 0; i < L / 4; i++) {
        const int q = (kgroup0 >> 2) + i;
        put4(b + (q >> 1) * HALF_B + (tid % BN) * 16 + (q & 1) * 8, PLANE_B, s.b[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < CPP; i++) put4(b + (bkq >> 1) * HALF_B + (bcol + i) * 16 + (bkq & 1) * 8, PLANE_B, s.b[i]);
    }
  };

  f32x16 acc[MT][NT], small[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[a][b][r] = small[a][b][r] = 0.0f;

  auto compute = [&](const unsigned char *buf) {
    const unsigned char *const fa = buf + half * HALF_A + (wrow + li) * 16;
    const unsigned char *const fb = buf + 3 * PLANE_A + half * HALF_B + (wcol + li) * 16;
    bf16x8 a[MT][3], b[NT][3];
#pragma unroll
    for (int pl = 0; pl < 3; pl++) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++) a[mt][pl] = *reinterpret_cast<const bf16x8 *>(fa + pl * PLANE_A + mt * 512);
#pragma unroll
      for (int nt = 0; nt < NT; nt++) b[nt][pl] = *reinterpret_cast<const bf16x8 *>(fb + pl * PLANE_B + nt * 512);
    }
    auto products = [&](int i, int j, f32x16 (&sum)[MT][NT]) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
          sum[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[mt][i], b[nt][j], sum[mt][nt], 0, 0, 0);
    };
    products(0, 0, acc);
    products(0, 1, small);
    products(1, 0, small);
    products(1, 1, small);
    products(0, 2, small);
    products(2, 0, small);
  };

  // Slab s+2 is requested, slab s+1 split and stored to the other LDS buffer, slab s multiplied: one barrier a slab.
  const int nslabs = (kshare + BK - 1) / BK, nfull = kend > kbeg ? (kend - kbeg) / BK : 0;
  Slab next;
  read_taps(kbeg);
  fetch(kbeg, next, true);
  put(lds[0], next);
  if (nslabs > 1) fetch(kbeg + BK, next, true);
  __syncthreads();
  auto step = [&](int s, int cur) {
    const Slab now = next;
    fetch(kbeg + (s + 2) * BK, next, false);
    __builtin_amdgcn_s_setprio(1);
    compute(lds[cur]);
    put(lds[cur ^ 1], now);
    // fragment reads, requests, then products with the split and the stores in between
    constexpr int PIECES = NA + (B_IS_KC ? NB : (IM2COL ? L / 4 : CPP));
    constexpr int PRODUCTS = MT * NT * 6, VALU = PIECES * (BY_PAIR ? 26 : 28) + (IM2COL ? 2 * L : 0), STORES = PIECES * 3;
    constexpr int LOADS = NA + (B_IS_KC ? NB : (IM2COL ? L : PIX_ANY ? 4 * CPP : 4));
    __builtin_amdgcn_sched_group_barrier(0x100, (MT + NT) * 3, 0);
    __builtin_amdgcn_sched_group_barrier(0x20, LOADS, 0);
#pragma unroll
    for (int i = 0; i < PRODUCTS; i++) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, (VALU + PRODUCTS - 1) / PRODUCTS, 0);
      if ((i + 1) * STORES / PRODUCTS > i * STORES / PRODUCTS) __builtin_amdgcn_sched_group_barrier(0x200, (STORES + PRODUCTS - 1) / PRODUCTS, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
  };
  int s = 0;
  // (every group takes the barriers of the one that has most)
  for (const int nall = KG == 1 ? nfull : (klast - kfirst - (KG - 1) * kshare) / BK; s + 3 < nall; s += 2) {
    step(s, 0);
    step(s + 1, 1);
  }
  for (; s < nslabs; s++) {
    const Slab now = next;
    if (s + 2 < nslabs) fetch(kbeg + (s + 2) * BK, next, true);
    compute(lds[s & 1]);
    if (s + 1 < nslabs) put(lds[(s & 1) ^ 1], now);
    __syncthreads();
  }

  // ---- the two sums meet; is there anything the split could not hold? ------------------------------------
  SumRange sums = {0xffffffffu, 0};
#pragma unroll
  for (int b = 0; b < NT; b++) {
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[a][b][r] += small[a][b][r];
    if (!CONV && !B_IS_KC && col0 + wcol + b * 32 + li >= p.n) continue;  // (zeros; elsewhere surplus columns repeat the last ones)
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int r = 0; r < 16; r++) add_sum(sums, acc[a][b][r]);
  }
  bool again = __syncthreads_or(not_finite(sums) || lost || loses_bits(least));
  if (again && !__syncthreads_or(not_finite(sums) || small_sums(sums))) {
    // (elements that lost bits, but every sum is large: what were their partners?)
    bool large = false;
    read_taps(kbeg);
    constexpr int AHEAD = IM2COL ? 1 : 2;
    for (int k0 = kbeg; k0 < kend; k0 += AHEAD * BK) {
      Slab q[AHEAD];
#pragma unroll
      for (int i = 0; i < AHEAD; i++) fetch(k0 + i * BK, q[i], true);
#pragma unroll
      for (const Slab &s : q) {
#pragma unroll
        for (const f32x4 &v : s.a) large |= reaches_partners(v);
#pragma unroll
        for (const f32x4 &v : s.b) large |= reaches_partners(v);
      }
    }
    again = __syncthreads_or(large);
  }
  if (KG > 1 && !again) {
    // sums of the groups behind the first, in order; each through its own LDS
    float *const mine = reinterpret_cast<float *>(&lds[0][0]);
    if (group > 0) {
#pragma unroll
      for (int a = 0; a < MT; a++)
#pragma unroll
        for (int b = 0; b < NT; b++)
#pragma unroll
          for (int r = 0; r < 16; r++) mine[((a * NT + b) * 16 + r) * THREADS + tid] = acc[a][b][r];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KG; g++) {
      const float *const other = reinterpret_cast<const float *>(&lds_all[g][0][0]);
#pragma unroll
      for (int a = 0; a < MT; a++)
#pragma unroll
        for (int b = 0; b < NT; b++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[a][b][r] += other[((a * NT + b) * 16 + r) * THREADS + tid];
    }
  }
  if (again) {
    if (group > 0) return;  // (the first group does the whole K again)
    // The same slabs through the same LDS, whole: [row or column][16 k, 4 apart]; a lane multiplies eight neighbouring k.
    // (us, fp32 instruction / a NaN in every row: 4096^3 940 / 1586, 4096x3072x768 146 / 273, 1024^3 36 / 44; with loads of
    // single elements 4089, 605, 128.)
    constexpr int LDW = BK + 4;
    static_assert((BM + BN) * LDW * 4 <= BUF, "whole slabs");
    auto put_whole = [&](float *buf, const Slab &s) {
      float *const b = buf + BM * LDW;
#pragma unroll
      for (int i = 0; i < NA; i++) *reinterpret_cast<f32x4 *>(buf + ((tid >> 2) + i * RPP) * LDW + kq * 4) = s.a[i];
#pragma unroll
      for (int i = 0; i < (B_IS_KC ? NB : (IM2COL ? L / 4 : CPP)); i++) {
        const int col = B_IS_KC ? (tid >> 2) + i * RPP : (IM2COL ? tid % BN : bcol + i);
        const int q = B_IS_KC ? kq : (IM2COL ? (kgroup0 >> 2) + i : bkq);
        *reinterpret_cast<f32x4 *>(b + col * LDW + q * 4) = s.b[i];
      }
    };
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < NT; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
    kend = klast;  // (of group 0, which begins with the tile's first slab)
    read_taps(kfirst);
    fetch(kfirst, next, true);
    for (int k0 = kfirst, cur = 0; k0 < klast; k0 += BK, cur ^= 1) {
      float *const buf = reinterpret_cast<float *>(&lds[cur][0]);
      put_whole(buf, next);
      if (k0 + BK < klast) fetch(k0 + BK, next, true);
      __syncthreads();
      const float *const fa = buf + (wrow + li) * LDW + 8 * half, *const fb = buf + (BM + wcol + li) * LDW + 8 * half;
      f32x4 a[MT][2], b[NT][2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) a[mt][h] = *reinterpret_cast<const f32x4 *>(fa + mt * 32 * LDW + 4 * h);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) b[nt][h] = *reinterpret_cast<const f32x4 *>(fb + nt * 32 * LDW + 4 * h);
      }
#pragma unroll
      for (int e = 0; e < 8; e++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int nt = 0; nt < NT; nt++)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[mt][e >> 2][e & 3], b[nt][e >> 2][e & 3], acc[mt][nt], 0, 0, 0);
    }
    __syncthreads();  // (the epilogue's staging is this LDS)
  }
  finish_tile<BM, BN, WM, WN, CONV, (MT * NT > 2 ? 2 : 1)>(p, acc, tw.whole, tw.lin, tw.chunk, bz, row0, col0,
                                    reinterpret_cast<float *>(&lds[0][0]) + wave * STAGE_FLOATS);
}

template <int BM, int BN, int WM, int WN, int BMODE, int KG>
__global__ __launch_bounds__(WM * WN * 64 * KG, split_blocks(BM, BN)) void split_kernel(Params p) {
  split_tile<BM, BN, WM, WN, BMODE, KG>(p, (int)blockIdx.x);
}

// Several independent products in one launch: the tiles of problem i follow those of problem i - 1.
template <int BMODE, int KG>
__global__ __launch_bounds__(256 * KG, split_blocks(64, 64)) void split_group_kernel(GroupParams g) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < GROUP_MAX; j++)
    if (j < g.count && (int)blockIdx.x >= g.first[j]) i = j;
  split_tile<64, 64, 2, 2, BMODE, KG>(g.p[i], (int)blockIdx.x - g.first[i]);
}

template <int BM, int BN, int WM, int WN, int BMODE, int KG = 1>
int launch_split_tile(Params &p, int nz, const WorkPlan &w) {
  if (BMODE != B_PIXELS_ANY) g_last_form = BMODE;  // (otherwise the caller says which conv it is)
  return launch_planned<BM, BN>(p, nz, BMODE >= B_IM2COL32, BK, 0, [&](dim3 grid, bool) {
    hipLaunchKernelGGL((split_kernel<BM, BN, WM, WN, BMODE, KG>), grid, dim3(WM * WN * 64 * KG), 0, wdh::stream(), p);
  }, &w);
}
template <int BMODE>
int launch_split(const SplitPlan &s, Params &p, int nz) {
  switch (s.tile) {
    case S256x128:
      if constexpr (BMODE == B_KC || BMODE == B_MC) return launch_split_tile<256, 128, 4, 2, BMODE>(p, nz, s.work);
      [[fallthrough]];  // (not planned for convs)
    case S128x128: return launch_split_tile<128, 128, 2, 2, BMODE>(p, nz, s.work);
    case S64x128: return launch_split_tile<64, 128, 2, 2, BMODE>(p, nz, s.work);
    case S128x64: return launch_split_tile<128, 64, 2, 2, BMODE>(p, nz, s.work);
    case S64x64K2: return launch_split_tile<64, 64, 2, 2, BMODE, 2>(p, nz, s.work);
    case S64x64K4: return launch_split_tile<64, 64, 2, 2, BMODE, 4>(p, nz, s.work);
    default: return launch_split_tile<64, 64, 2, 2, BMODE>(p, nz, s.work);
  }
}

}  // namespace wdhc

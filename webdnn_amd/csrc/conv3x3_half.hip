// 3x3, stride-1, undilated, ungrouped convolutions of a batch on the f16 matrix cores, straight from the input: products of two f16
// parts each (half_product.h says what they hold, how they are added up and what is done again) in the arrangement of
// conv3x3_split.hip, input rows in LDS, split once per tile, weights packed beforehand.
//
// K runs over blocks of 16 input channels, and within a block over pairs of taps: one v_mfma_f32_16x16x32_f16 multiplies
// sixteen channels of two taps, lanes 0 to 31 having the first tap and 32 to 63 the second; the ninth tap has a step to itself, against
// zeros (a tenth of the products).  Blocks of 32 channels would not need it, but their next rows would take 60 registers on the way.
// Sums leave the accumulators every two steps, and the weights of a pair of steps are requested two pairs ahead.
//
// Bound: as half_product.h; a block takes 2.7 us on a CU by itself, 4.3 when all have one, where its products alone take 1.6.
// (us, bfloat16 parts or transforms / this: 32 images 128 -> 128 on 28x28 55 / 36 to 41, 128 images 150 / 119, 256 -> 256 on 14x14
// 151 / 115, 64 images 208 -> 608 on 20x20 116 / 89.)  A wavefront with 128 pixels instead of 64 spills 100 registers.
#include "half_product.h"

namespace wdhc {

constexpr int CB = 16;          // channels per block
constexpr int KGRAN = CB * 9;   // k per block
constexpr int most_of(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }

// WP x WQ wavefronts of 32 output channels x 128 / WQ pixels; KG groups of them share the channels.
// BUFS: LDS buffers for blocks of channels.  Two where they fit: the next block is stored between this one's products.
template <int WP, int WQ, int KG, int PX, int BUFS>
__global__ __launch_bounds__(WP * WQ * KG * 64, 2) void conv3x3_half_kernel(Params p, HalfOperand w) {
  constexpr int THREADS = WP * WQ * 64, BM = WP * 32, BN = 128, QC = BN / WQ, QB = QC / 16;
  constexpr int XU = (2 * PX + THREADS - 1) / THREADS;  // (pixel slot, channel eight) items per thread
  constexpr int EIGHT = PX * 16, PART = 2 * EIGHT, BUF = 2 * PART, SUMS = BM * BN * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[most_of(KG * BUFS * BUF, (KG - 1) * SUMS, WP * WQ * STAGE_FLOATS * 4)];
  __shared__ unsigned most[KG * WP * WQ];

  const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);
  unsigned char *const xs = lds + group * BUFS * BUF;
  const int tid = (int)threadIdx.x - group * THREADS;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave / WQ, wq = wave % WQ;
  const int c16 = lane & 15, g4 = lane >> 4;
  const ConvGeom &cv = p.cv;
  const int plane_in = cv.h * cv.w;

  const TileWork tw = decode_work(p, (int)blockIdx.x);
  const int row0 = tw.tm * BM, col0 = tw.tn * BN;
  const int kfirst = tw.whole ? 0 : tw.chunk * p.kchunk;
  const int klast = tw.whole ? p.k : (kfirst + p.kchunk < p.k ? kfirst + p.kchunk : p.k);
  const int kshare = ((klast - kfirst) / KGRAN + KG - 1) / KG * KGRAN;
  const int kbeg = kfirst + group * kshare, kend = kbeg + kshare < klast ? kbeg + kshare : klast;

  // ---- the tile's input rows: slot -> (image, row), as in conv3x3_halo_kernel ------------------------------
  const int R0 = fdiv(col0, cv.fd_ow), img0 = fdiv(R0, cv.fd_oh);
  const int first_rows = (img0 + 1) * cv.oh - R0;  // output rows from R0 to the end of its image
  const int npx = cv.slots * cv.pitch;
  int voff_x[XU], lds_x[XU];
#pragma unroll
  for (int i = 0; i < XU; i++) {
    const int u = tid + THREADS * i;
    const int ch = u >= npx ? 1 : 0, px = u - ch * npx;
    const int slot = fdiv(px, cv.fd_pg), cx = px - slot * cv.pitch;
    int d, iy;
    if (slot < first_rows + 2) {
      d = 0;
      iy = (R0 - img0 * cv.oh) - cv.pt + slot;
    } else {
      const int s2 = slot - first_rows - 2, dd = fdiv(s2, cv.fd_oh2);
      d = 1 + dd;
      iy = s2 - dd * (cv.oh + 2) - cv.pt;
    }
    const int img = img0 + d, ix = cx - cv.pl;
    const bool live = u < 2 * npx;
    const bool data = live && (long long)img * cv.oh * cv.ow < cv.npix && iy >= 0 && iy < cv.h && ix >= 0 && ix < cv.w;
    voff_x[i] = data ? (((img * cv.c_total + 8 * ch) * cv.h + iy) * cv.w + ix) * 4 : BUF_OOB;
    lds_x[i] = live ? ch * EIGHT + px * 16 : -1;
  }
  const rsrc_t rsrc_x = make_rsrc(p.B, p.b_bytes);
  // where the corner of a pixel lies
  auto corner_of = [&](int P) {
    P = P < (int)cv.npix ? P : (int)cv.npix - 1;  // lanes past the edge are never stored
    const int R = fdiv(P, cv.fd_ow), ox = P - R * cv.ow;
    const int slot0 = (R - R0) + 2 * (fdiv(R, cv.fd_oh) - img0);
    return (slot0 * cv.pitch + ox) * 16;
  };
  int corner[QB], shift[5];  // (a step is two taps, of which a lane has one; the last step has one for all)
#pragma unroll
  for (int j = 0; j < QB; j++) corner[j] = (g4 & 1) * EIGHT + corner_of(col0 + wq * QC + 16 * j + c16);
#pragma unroll
  for (int s = 0; s < 5; s++) {
    const int tap = s < 4 ? 2 * s + (g4 >> 1) : 8;
    shift[s] = (tap / 3 * cv.pitch + tap % 3) * 16;
  }

  float x[XU][8];
  auto fetch_item = [&](int k0, int i) {  // of the block of channels that begins at k0
    const int v = k0 < kend ? voff_x[i] : BUF_OOB, soff = k0 / 9 * plane_in * 4;
#pragma unroll
    for (int j = 0; j < 8; j++) x[i][j] = buf_load(rsrc_x, v, soff + j * plane_in * 4);
  };
  auto fetch_x = [&](int k0) {
#pragma unroll
    for (int i = 0; i < XU; i++) fetch_item(k0, i);
  };
  float sq = 1.0f;
  auto put_item = [&](unsigned char *buf, int i) {
    const HalfParts q = half_parts(x[i], sq);
    if (lds_x[i] >= 0) {
      *reinterpret_cast<f16x8 *>(buf + lds_x[i]) = q.h;
      *reinterpret_cast<f16x8 *>(buf + lds_x[i] + PART) = q.l;
    }
  };
  auto put_x = [&]() {
#pragma unroll
    for (int i = 0; i < XU; i++) put_item(xs, i);
  };

  // ---- the weights: from L2 straight into the lanes, two steps at a time (the last of a block by itself) ----------
  const rsrc_t rsrc_p = make_rsrc(w.packed, (int)half_fragment_bytes(w.strips, w.steps));
  const int strip0 = row0 / 16 + wp * 2, stripsize = w.steps * STEP_BYTES;
  struct Strips { f16x8 h[2][2], l[2][2]; } pair[3];  // [strip][step]
  auto fetch_strips = [&](int k0, int pi, Strips &s) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // (past the last strip, or the last block: some other one again, as in half_product.h)
      const int strip = strip0 + i < w.strips ? strip0 + i : w.strips - 1, block = k0 < p.k ? k0 / KGRAN : 0;
      const int soff = strip * stripsize + (block * 5 + 2 * pi) * STEP_BYTES;
#pragma unroll
      for (int t = 0; t < (pi < 2 ? 2 : 1); t++) {
        s.h[i][t] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, lane * 16, soff + t * STEP_BYTES, 0));
        s.l[i][t] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, lane * 16 + 1024, soff + t * STEP_BYTES, 0));
      }
    }
  };

  f32x4 total[2][QB];  // [strip][16 pixels]
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < QB; j++) total[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // the first block says what the others are scaled by
  fetch_x(kbeg);
  fetch_strips(kbeg, 0, pair[0]);
  fetch_strips(kbeg, 1, pair[1]);
  unsigned top = 0;
#pragma unroll
  for (int i = 0; i < XU; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const unsigned u = __float_as_uint(x[i][j]) & 0x7fffffffu;
      top = u > top ? u : top;
    }
  const int eq = __builtin_amdgcn_readfirstlane(scale_exponent(group_most<WP * WQ>(top, most + group * WP * WQ, wave), X_TARGET));
  sq = scale_of(eq);
  put_x();
  fetch_x(kbeg + KGRAN);
  __syncthreads();

  struct Columns { f16x8 h[2], l[2]; } columns[2];  // [step of the pair]
  auto read_columns = [&](int buf, int pi, int j, Columns &c) {
#pragma unroll
    for (int t = 0; t < (pi < 2 ? 2 : 1); t++) {
      const unsigned char *const at = xs + buf + corner[j] + shift[2 * pi + t];
      c.h[t] = *reinterpret_cast<const f16x8 *>(at);
      c.l[t] = *reinterpret_cast<const f16x8 *>(at + PART);
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
  const int blocks = kshare / KGRAN;
  if (BUFS > 1) read_columns(0, 0, 0, columns[0]);
  for (int b = 0, cur = 0; b < blocks; b++, cur = BUFS > 1 ? BUF - cur : 0) {
    const int k0 = kbeg + b * KGRAN;
    if (BUFS == 1) read_columns(0, 0, 0, columns[0]);
#pragma unroll
    for (int pi = 0; pi < 3; pi++) {
      const Strips &s = pair[pi];
      // what the pair before this one was multiplied with is requested anew: two pairs ahead
      if (pi == 0) fetch_strips(k0, 2, pair[2]);
      else fetch_strips(k0 + KGRAN, pi - 1, pair[pi - 1]);
#pragma unroll
      for (int j = 0; j < QB; j++) {
        const Columns &c = columns[j & 1];
        if (j + 1 < QB) {
          read_columns(cur, pi, j + 1, columns[(j + 1) & 1]);
        } else if (pi < 2) {
          read_columns(cur, pi + 1, 0, columns[0]);
        } else if (BUFS > 1) {
          __syncthreads();
          read_columns(BUF - cur, 0, 0, columns[0]);
        }
        f32x4 h[2], l[2];
        auto products = [&](const f16x8 (&a)[2][2], int t, f16x8 q, f32x4 (&sum)[2], bool first) {
#pragma unroll
          for (int i = 0; i < 2; i++) sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][t], q, first ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : sum[i], 0, 0, 0);
        };
        products(s.h, 0, c.l[0], l, true);
        products(s.h, 0, c.h[0], h, true);
        products(s.l, 0, c.h[0], l, false);
        if (pi < 2) {
          products(s.h, 1, c.h[1], h, false);
          products(s.h, 1, c.l[1], l, false);
          products(s.l, 1, c.h[1], l, false);
        }
        flush((j + QB - 1) % QB);
        const int item = pi * QB + j - 1;  // (stored behind the first group of a block)
        const bool puts = BUFS > 1 && pi < 2 && item >= 0 && item < XU;
        if (puts) {
          put_item(xs + BUF - cur, item);
          fetch_item(k0 + 2 * KGRAN, item);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) high[i] = h[i], low[i] = l[i];
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 12; i++) {
          if (pi == 2 && i >= 6) continue;
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          if (puts) __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
          else if (pi == 2) __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
          else __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (BUFS == 1 && b + 1 < blocks) {
      __syncthreads();  // everybody has read the block before
      put_x();
      fetch_x(k0 + 2 * KGRAN);
      __syncthreads();
    }
  }
  flush(QB - 1);

  // ---- unscaled; is there anything the two parts could not hold? ------------------------------------------
  const HalfDoubt doubt = unscale<true, QB>(total, w, strip0, p.m, eq);
  bool again = false;
  if (__syncthreads_or(doubt.bad || doubt.tiny)) {
    again = __syncthreads_or(doubt.bad);
    if (!again) {
      unsigned *const lossy = reinterpret_cast<unsigned *>(xs);
      if (tid == 0) lossy[0] = 0;
      __syncthreads();
      const float least = __builtin_ldexpf(1.0f, FULL_EXPONENT - eq);
      unsigned count = 0;
      for (int k0 = kbeg; k0 < kend; k0 += KGRAN) {
        fetch_x(k0);
#pragma unroll
        for (int i = 0; i < XU; i++)
#pragma unroll
          for (int j = 0; j < 8; j++) count += __builtin_fabsf(x[i][j]) < least && x[i][j] != 0.0f ? 9u : 0u;
      }
      if (count) atomicAdd(&lossy[0], count);
      __syncthreads();
      again = __syncthreads_or(kend > kbeg && shows_loss<true, QB>(total, w, lossy, 0, strip0, p.m, col0 + wq * QC, p.n, eq, kend - kbeg));
    }
  }
  f32x16 acc[1][QC / 32];
  to_blocks<true, QB>(total, acc);
  if (KG > 1 && !again && !join_groups<KG, THREADS>(acc, lds, SUMS, group, tid)) return;
  if (again) {
    if (group > 0) return;
    // The same rows through the same LDS, whole: [channel eight][pixel][8 channels]; the weights as the caller has them.
    const int li = lane & 31, half = lane >> 5;
    constexpr int NT = QC / 32;
    int at[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      at[nt] = half * 2 * EIGHT + 2 * corner_of(col0 + wq * QC + nt * 32 + li);
#pragma unroll
      for (int r = 0; r < 16; r++) acc[0][nt][r] = 0.0f;
    }
    const int r0 = row0 + wp * 32 + li;
    const float *const wt = p.A + (long long)(r0 < p.m ? r0 : p.m - 1) * p.k + 72 * half;
    for (int k0 = kfirst; k0 < klast; k0 += KGRAN) {
      const int soff = k0 / 9 * plane_in * 4;
#pragma unroll
      for (int i = 0; i < XU; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) x[i][j] = buf_load(rsrc_x, voff_x[i], soff + j * plane_in * 4);
      __syncthreads();  // everybody has read the block before
#pragma unroll
      for (int i = 0; i < XU; i++)
        if (lds_x[i] >= 0) {
          f32x4 *const cell = reinterpret_cast<f32x4 *>(xs + 2 * lds_x[i]);
          cell[0] = f32x4{x[i][0], x[i][1], x[i][2], x[i][3]};
          cell[1] = f32x4{x[i][4], x[i][5], x[i][6], x[i][7]};
        }
      __syncthreads();
#pragma unroll 1
      for (int tap = 0; tap < 9; tap++) {
        const int off = (tap / 3 * cv.pitch + tap % 3) * 32;
        float ea[8];
        f32x4 eb[NT][2];
#pragma unroll
        for (int j = 0; j < 8; j++) ea[j] = wt[k0 + j * 9 + tap];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
          const f32x4 *const cell = reinterpret_cast<const f32x4 *>(xs + at[nt] + off);
          eb[nt][0] = cell[0];
          eb[nt][1] = cell[1];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
          for (int nt = 0; nt < NT; nt++)
            acc[0][nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ea[j], eb[nt][j >> 2][j & 3], acc[0][nt], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  finish_tile<BM, BN, WP, WQ, true, 2>(p, acc, tw.whole, tw.lin, tw.chunk, 0, row0, col0, reinterpret_cast<float *>(lds) + wave * STAGE_FLOATS);
}

template <int WP, int WQ, int KG, int PX, int BUFS>
static int launch_one(Params &p, const HalfOperand &w, const WorkPlan &work) {
  g_last_form = WDH_FORM_CONV3X3_LDS;
  return launch_planned<WP * 32, 128>(p, 1, true, KGRAN, 0, [&](dim3 grid, bool) {
    hipLaunchKernelGGL((conv3x3_half_kernel<WP, WQ, KG, PX, BUFS>), grid, dim3(WP * WQ * KG * 64), 0, wdh::stream(), p, w);
  }, &work);
}
template <int PX>
static int launch_tile(Params &p, const HalfPlan &s, const HalfOperand &w) {
  switch (s.tile) {
    case H3_128: return launch_one<4, 2, 1, PX, 2>(p, w, s.work);
    case H3_64: return launch_one<2, 2, 1, PX, (PX <= 480 ? 2 : 1)>(p, w, s.work);
    default: return launch_one<2, 2, 2, PX, (PX <= 480 ? 2 : 1)>(p, w, s.work);
  }
}
int launch_conv3x3_half(Params &p, const HalfPlan &s, const HalfOperand &w) {
  return p.cv.slots * p.cv.pitch > 480 ? launch_tile<640>(p, s, w) : launch_tile<480>(p, s, w);
}

}  // namespace wdhc

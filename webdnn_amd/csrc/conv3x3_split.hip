// 3x3, stride-1, undilated, ungrouped convolutions of a batch on the bf16 matrix cores, straight from the input: every
// input element is fetched and split into its three bfloat16 parts (split_product.h) once per tile, not once per tap, and the
// weights arrive split.
//
// K runs over blocks of 16 input channels, and within a block over the nine taps: one tap of a block is one
// v_mfma_f32_32x32x16_bf16 step.  For a block the workgroup stages the input rows its BN output pixels touch in LDS,
// [h, m, l][channel half][pixel][8 channels]: a lane's fragment of a tap is one 16-byte read at a fixed distance
// from its pixel's corner, neighbouring lanes side by side.  Rows and columns of padding are slots that are filled with zeros
// (loads outside the descriptor).  The weights are laid out fragment by fragment beforehand (pack_kernel; kept per weight
// buffer when the caller vouches for it), [32 rows][block, tap][h, m, l][lane][8 channels], and go from L2 straight into registers.
// Behind them a word for each [32 rows][block, tap] says what the split has to know of its weights (WEIGHTS_*).
#include <string.h>

#include "split_product.h"

namespace wdhc {

constexpr int CB = 16;          // channels per block
constexpr int KGRAN = CB * 9;   // k per block
constexpr unsigned WEIGHTS_LOSE = 1, WEIGHTS_LARGE = 2;  // some lose bits; some reach 2^30 (split_product.h)
__host__ __device__ constexpr long long fragment_bytes(long long rows, long long steps) { return (rows + 31) / 32 * steps * 3072; }

// One thread: one lane's eight channels of one (row block, channel block, tap).
__global__ __launch_bounds__(256) void pack3x3_kernel(const float *__restrict__ W, u32x4 *__restrict__ P, int cout, int c) {
  const int steps = c / CB * 9;
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  const int lane = (int)(id & 63);
  const long long at = id >> 6;  // row block * steps + step
  if (at >= (long long)((cout + 31) / 32) * steps) return;
  const int rb = (int)(at / steps), step = (int)(at - (long long)rb * steps);
  const int row = rb * 32 + (lane & 31), c0 = step / 9 * CB + 8 * (lane >> 5), tap = step % 9;
  float w[8];
#pragma unroll
  for (int j = 0; j < 8; j++) w[j] = row < cout ? W[((long long)row * c + c0 + j) * 9 + tap] : 0.0f;
  unsigned least = 0xffffffffu;
  bool large = false;
#pragma unroll
  for (int j = 0; j < 8; j++) large |= reaches_partners(w[j]);
  u32x4 h, m, l;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const SplitPair s = split_pair(w[2 * j], w[2 * j + 1]);
    least = least_of(least, w[2 * j], w[2 * j + 1]);
    h[j] = s.h;
    m[j] = s.m;
    l[j] = s.l;
  }
  const unsigned word = (__any(loses_bits(least)) ? WEIGHTS_LOSE : 0) | (__any(large) ? WEIGHTS_LARGE : 0);
  if (lane == 0) reinterpret_cast<unsigned *>(reinterpret_cast<char *>(P) + fragment_bytes(cout, steps))[at] = word;
  u32x4 *const p = P + at * 192 + lane;
  p[0] = h;
  p[64] = m;
  p[128] = l;
}

template <int BM, int BN, int WM, int WN, int PX>
__global__ __launch_bounds__(WM * WN * 64, BM * BN >= 128 * 128 ? 2 : PX <= 480 ? 3 : 2) void conv3x3_split_kernel(Params p, const u32x4 *packed) {
  constexpr int THREADS = WM * WN * 64;
  constexpr int MT = BM / (WM * 32), NT = BN / (WN * 32);
  constexpr int XU = (2 * PX + THREADS - 1) / THREADS;  // (pixel slot, channel half) items per thread
  constexpr int HALF_X = PX * 16, PLANE_X = 2 * HALF_X;
  __shared__ __attribute__((aligned(16))) unsigned char xs[3 * PLANE_X];
  static_assert(3 * PLANE_X >= WM * WN * STAGE_FLOATS * 4, "epilogue staging");

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 31, half = lane >> 5;
  const int wrow = wm * (MT * 32), wcol = wn * (NT * 32);
  const ConvGeom &cv = p.cv;
  const int plane_in = cv.h * cv.w;

  const TileWork tw = decode_work(p, (int)blockIdx.x);
  const int row0 = tw.tm * BM, col0 = tw.tn * BN;
  const int kbeg = tw.whole ? 0 : tw.chunk * p.kchunk;
  const int kend = tw.whole ? p.k : (kbeg + p.kchunk < p.k ? kbeg + p.kchunk : p.k);

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
    lds_x[i] = live ? ch * HALF_X + px * 16 : -1;
  }
  const rsrc_t rsrc_x = make_rsrc(p.B, p.b_bytes);
  const int steps = p.k / CB;  // (block, tap) steps of a row block
  const rsrc_t rsrc_a = make_rsrc(packed, (int)fragment_bytes(p.m, steps));

  // where a lane finds the corner of its pixels, and its row blocks' weights
  int corner[NT], voff_a[MT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    int P = col0 + wcol + nt * 32 + li;
    P = P < (int)cv.npix ? P : (int)cv.npix - 1;  // lanes past the edge are never stored
    const int R = fdiv(P, cv.fd_ow), ox = P - R * cv.ow;
    const int slot0 = (R - R0) + 2 * (fdiv(R, cv.fd_oh) - img0);
    corner[nt] = half * HALF_X + (slot0 * cv.pitch + ox) * 16;
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    int rb = (row0 + wrow) / 32 + mt;
    rb = rb < (p.m + 31) / 32 ? rb : (p.m + 31) / 32 - 1;
    voff_a[mt] = rb * steps * 3072 + lane * 16;
  }

  f32x16 acc[MT][NT], small[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[a][b][r] = small[a][b][r] = 0.0f;

  // what is known of the weights of this tile and chunk
  auto weights_have = [&](unsigned what) {
    const unsigned *const words = reinterpret_cast<const unsigned *>(reinterpret_cast<const char *>(packed) + fragment_bytes(p.m, steps));
    const int count = (kend - kbeg) / CB;
    unsigned w = 0;
#pragma unroll
    for (int i = 0; i < BM / 32; i++)
      if (row0 + 32 * i < p.m)
        for (int j = tid; j < count; j += THREADS) w |= words[(row0 / 32 + i) * steps + kbeg / CB + j];
    return __any((w & what) != 0);
  };
  bool lost = false;  // whether this wavefront has met elements that lose bits

  float x[XU][8];
  auto fetch_x = [&](int k0) {  // the block of channels that begins at k0
    const int soff = k0 / 9 * plane_in * 4;
#pragma unroll
    for (int i = 0; i < XU; i++)
#pragma unroll
      for (int j = 0; j < 8; j++) x[i][j] = buf_load(rsrc_x, voff_x[i], soff + j * plane_in * 4);
  };
  auto put_x = [&]() {
    unsigned least = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < XU; i++) {
      u32x4 h, m, l;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const SplitPair s = split_pair(x[i][2 * j], x[i][2 * j + 1]);
        least = least_of(least, x[i][2 * j], x[i][2 * j + 1]);
        h[j] = s.h;
        m[j] = s.m;
        l[j] = s.l;
      }
      if (lds_x[i] >= 0) {
        *reinterpret_cast<u32x4 *>(xs + lds_x[i]) = h;
        *reinterpret_cast<u32x4 *>(xs + lds_x[i] + PLANE_X) = m;
        *reinterpret_cast<u32x4 *>(xs + lds_x[i] + 2 * PLANE_X) = l;
      }
    }
    lost |= __any(loses_bits(least));
  };
  struct Frags { bf16x8 a[MT][3], b[NT][3]; };
  auto fetch_a = [&](int step, Frags &f) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int pl = 0; pl < 3; pl++)
        f.a[mt][pl] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, voff_a[mt], step * 3072 + pl * 1024, 0));
  };
  auto read_b = [&](int tap, Frags &f) {
    const int shift = ((tap / 3) * cv.pitch + tap % 3) * 16;
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int pl = 0; pl < 3; pl++) f.b[nt][pl] = *reinterpret_cast<const bf16x8 *>(xs + corner[nt] + shift + pl * PLANE_X);
  };
  auto products = [&](const Frags &f, int i, int j, f32x16 (&sum)[MT][NT]) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
        sum[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[mt][i], f.b[nt][j], sum[mt][nt], 0, 0, 0);
  };

  Frags f[2];
  fetch_x(kbeg);
  fetch_a(kbeg / CB, f[0]);
  lost = weights_have(WEIGHTS_LOSE);
  for (int k0 = kbeg; k0 < kend; k0 += KGRAN) {
    if (k0 != kbeg) __syncthreads();  // everybody has read the block before
    put_x();
    __syncthreads();
    if (k0 + KGRAN < kend) fetch_x(k0 + KGRAN);
    const int step0 = k0 / CB;
    read_b(0, f[0]);
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
      Frags &now = f[tap & 1], &next = f[(tap + 1) & 1];
      if (tap < 8) {
        fetch_a(step0 + tap + 1, next);
        read_b(tap + 1, next);
      }
      products(now, 0, 0, acc);
      products(now, 0, 1, small);
      products(now, 1, 0, small);
      products(now, 1, 1, small);
      products(now, 0, 2, small);
      products(now, 2, 0, small);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (k0 + KGRAN < kend) fetch_a(step0 + 9, f[0]);
  }

  // the two sums meet; what the split could not hold is done again (split_product.h)
  SumRange sums = {0xffffffffu, 0};
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        acc[a][b][r] += small[a][b][r];
        add_sum(sums, acc[a][b][r]);
      }
  bool again = __syncthreads_or(not_finite(sums) || lost);
  if (again && !__syncthreads_or(not_finite(sums) || small_sums(sums))) {
    bool large = weights_have(WEIGHTS_LARGE);
    for (int k0 = kbeg; k0 < kend; k0 += KGRAN) {
      fetch_x(k0);
#pragma unroll
      for (int i = 0; i < XU; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) large |= reaches_partners(x[i][j]);
    }
    again = __syncthreads_or(large);
  }
  if (again) {
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < NT; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
    // The same rows through the same LDS, whole: [channel half][pixel][8 channels]; the weights as the caller has them.
    const float *wt[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int r = row0 + wrow + mt * 32 + li;
      wt[mt] = p.A + (long long)(r < p.m ? r : p.m - 1) * p.k + 72 * half;
    }
    fetch_x(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += KGRAN) {
      __syncthreads();  // everybody has read the block before
#pragma unroll
      for (int i = 0; i < XU; i++)
        if (lds_x[i] >= 0) {
          f32x4 *const cell = reinterpret_cast<f32x4 *>(xs + 2 * lds_x[i]);
          cell[0] = f32x4{x[i][0], x[i][1], x[i][2], x[i][3]};
          cell[1] = f32x4{x[i][4], x[i][5], x[i][6], x[i][7]};
        }
      __syncthreads();
      if (k0 + KGRAN < kend) fetch_x(k0 + KGRAN);
#pragma unroll 1
      for (int tap = 0; tap < 9; tap++) {
        const int shift = (tap / 3 * cv.pitch + tap % 3) * 32;
        float ea[MT][8];
        f32x4 eb[NT][2];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int j = 0; j < 8; j++) ea[mt][j] = wt[mt][k0 + j * 9 + tap];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
          const f32x4 *const cell = reinterpret_cast<const f32x4 *>(xs + 2 * corner[nt] + shift);
          eb[nt][0] = cell[0];
          eb[nt][1] = cell[1];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ea[mt][j], eb[nt][j >> 2][j & 3], acc[mt][nt], 0, 0, 0);
      }
    }
    __syncthreads();  // (the epilogue's staging is this LDS)
  }
  // (LOOK 2 for two blocks a wavefront as well, which split_tile leaves at 1: the same or a little faster here, 128 images 64 -> 64
  // on 56x56 with a residual 178.8 us with 1, 175.5 with 2, without 159.2 / 157.6)
  finish_tile<BM, BN, WM, WN, true, 2>(p, acc, tw.whole, tw.lin, tw.chunk, 0, row0, col0,
                                    reinterpret_cast<float *>(xs) + wave * STAGE_FLOATS);
}

size_t packed3x3_bytes(int cout, int c) {
  const long long steps = c / CB * 9;
  return (size_t)(fragment_bytes(cout, steps) + ((cout + 31) / 32 * steps) * 4);
}

int pack3x3_launch(const float *W, void *P, int cout, int c) {
  const long long threads = (long long)((cout + 31) / 32) * (c / CB) * 9 * 64;
  hipLaunchKernelGGL(pack3x3_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, wdh::stream(), W, (u32x4 *)P, cout, c);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}

// Fills in the LDS layout for tiles of bn pixels; false: the rows are too wide.
bool conv3x3_split_fits(ConvGeom &cv, int bn, int images, int pr) {
  cv.pitch = cv.pl + cv.w + pr;
  int rows = 2 + (bn - 2) / cv.ow, imgs = 2 + (bn - 2) / (cv.oh * cv.ow);
  if (imgs > images) imgs = images;
  if (rows > images * cv.oh) rows = images * cv.oh;
  cv.slots = rows + 2 * imgs;
  cv.fd_oh2 = make_fastdiv(cv.oh + 2);
  cv.fd_pg = make_fastdiv(cv.pitch);
  return cv.slots * cv.pitch <= 640;
}

template <int BM, int WM, int PX>
static int launch_one(Params &p, const WorkPlan &w, const void *packed) {
  g_last_form = WDH_FORM_CONV3X3_LDS;
  return launch_planned<BM, 128>(p, 1, true, KGRAN, 0, [&](dim3 grid, bool) {
    hipLaunchKernelGGL((conv3x3_split_kernel<BM, 128, WM, 2, PX>), grid, dim3(WM * 128), 0, wdh::stream(), p, (const u32x4 *)packed);
  }, &w);
}
int launch_conv3x3_split(Params &p, const SplitPlan &s, const void *packed) {
  const bool wide = p.cv.slots * p.cv.pitch > 480;
  if (s.tile == S128x128) return wide ? launch_one<128, 2, 640>(p, s.work, packed) : launch_one<128, 2, 480>(p, s.work, packed);
  return wide ? launch_one<64, 2, 640>(p, s.work, packed) : launch_one<64, 2, 480>(p, s.work, packed);
}

}  // namespace wdhc

// softmax(alpha * Q K) V for a batch of heads in one launch.
//
// The reference has no such operator: it runs MatMul, Mul, Softmax, MatMul as four
// nodes (src/descriptor_runner/operators/cpu/operators/standard/matmul.ts:11-111,
// softmax.ts:34-57).  This kernel produces what that chain produces, with the same
// rounding points: scores rounded to fp32 after the scale, the row maximum subtracted,
// e^x in fp32, the fp32 row sum, every e scaled by the sum's reciprocal (as the
// Softmax kernel of this library does), and the second product accumulated in fp32.
// Only the order of the additions inside the two products and the row sum differs.
//
// A workgroup of eight or sixteen wavefronts owns 32 query rows of one head:
//   1. scores: Q and 32-key blocks of K go through LDS, each wavefront takes its blocks in turn
//      (v_mfma_f32_32x32x2_f32 over the head dimension) and, when all are done with K, writes
//      alpha * S to LDS, the whole 32 x keys block (keys <= 1024: 129 KB of the CU's 160 KB);
//   2. softmax: four (two) rows per wavefront, in place in LDS;
//   3. output: the keys are cut across the wavefronts in blocks of 32, each wavefront
//      accumulates its share of P V on the matrix cores, and the partial 32 x HD
//      blocks are added in wavefront order through LDS.
// Within a block of 32 keys (or of the head dimension) the two halves of a wavefront
// take the lower and the upper 16 indices, so that a lane reads 16 contiguous floats
// of Q, K and P (16-byte loads) where the MFMA's natural order would interleave them.
#include <math.h>

#include "common.h"
#include "rowmath.h"

namespace {

using namespace wdh::rowmath;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int ATT_ROWS = 32;
constexpr int ATT_MAX_KEYS = 1024;

struct AttParams {
  const float *Q, *K, *V;
  float *Y;
  int tq, tk;
  int pitch;        // floats per LDS row: >= keys rounded up to 32, pitch/4 odd
  int row_blocks;   // ceil(tq / 32)
  long long sQb, sQi, sKb, sKj, sVb, sVj, sYb, sYi;
  float alpha;
};

// ATT_WAVES wavefronts per workgroup: 16 for a head dimension of 32 (every phase is a chain of
// dependent steps per wavefront; twice the wavefronts halve each chain), 8 where a wavefront's
// registers hold less of K and V.
//
// Bound: latency -- a workgroup has a CU to itself and goes through its phases once.  So a wavefront asks for everything at
// once, and for no more than its keys: PER_WAVE blocks of 32 keys (at most 32 * ATT_WAVES * PER_WAVE keys), not always the blocks of
// 1024; V under the scores where the registers hold it beside them, else before the softmax.
// (us, always 1024 keys' loads / these: 12 heads of 64, 200 tokens 12.6 / 11.0, 384 16.7 / 15.9, 600 26.4 / 24.1; 16 of 64, 1024 tokens
// 80.8 / 67.6; 8 of 32, 100 keys 7.8 / 6.4, 300 11.3 / 9.4; 8 of 128, 128 keys 14.2 / 12.2.)
// And for whole rows: K and Q, whose rows the matrix instruction wants one to a lane, pass through LDS.  Loaded by the lanes that
// multiply them they are 16 bytes from 64 places, and a line is fetched again for each of its eight pieces.  (us, lane by lane / rows
// through LDS, same bits: 12 heads of 64, 200 tokens 11.6 / 10.7, 384 16.9 / 14.8, 600 26.1 / 22.7; 128 of 64, 384 105.7 / 88.6; 16 of 64, 1024
// 71.4 / 62.5; 8 of 32, 100 keys 6.9 / 6.8, 850 19.7 / 18.7; 128 of 32, 300 41.2 / 40.3; 8 of 128, 128 keys 12.7 / 11.8, 900 64.6 / 56.7.  Lane by
// lane with everything requested at once is slower than one piece after the other: 384 tokens 19.1.)  Of V a lane wants a column: its
// loads are whole rows as they are; they are asked for when the wavefront's first keys are in LDS and waited for where they multiply.
// Heads of 32 with one block a wavefront are held to 64 registers, so that two workgroups share a CU (512 heads, 100 keys 46.3 / 35.5).
template <int HD, int ATT_WAVES, int PER_WAVE>
__global__ __launch_bounds__(64 * ATT_WAVES, HD == 32 && PER_WAVE == 1 ? 8 : ATT_WAVES / 4) void attention_rows_kernel(AttParams p) {
  static_assert(HD % 32 == 0 && HD >= 32 && HD <= 128, "head dimension");
  static_assert(ATT_WAVES == 8 || ATT_WAVES == 16, "32 rows and the key blocks are dealt over the wavefronts");
  static_assert(32 * ATT_WAVES * PER_WAVE <= ATT_MAX_KEYS, "keys");
  constexpr int HALF = HD / 2;   // head-dimension indices per half wavefront
  constexpr int NB = HD / 32;    // 32-column blocks of the output
  constexpr int V_REGS = 16 * NB * PER_WAVE;
  constexpr bool V_FIRST = V_REGS <= 64, V_HELD = V_REGS <= 128;
  // Blocks beyond the keys are not asked for, except where most wavefronts have all of theirs anyway and the branches cost
  // more (us, asked for / left out: 8 heads of 32, 850 keys 18.1 / 18.7; 8 of 128, 900 keys 61 / 80; but 12 of 64, 600 keys 33.0 / 24.6).
  constexpr bool SKIP = HD == 64 || PER_WAVE == 1;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, half = lane >> 5;
  const int b = blockIdx.x / p.row_blocks;
  const int row0 = (blockIdx.x - b * p.row_blocks) * ATT_ROWS;
  const float *Q = p.Q + (long long)b * p.sQb;
  const float *K = p.K + (long long)b * p.sKb;
  const float *V = p.V + (long long)b * p.sVb;
  const int ncb = (p.tk + 31) >> 5;  // blocks of 32 keys

  // Every value of V this wavefront will need in step 3 (up to 64 registers travel while the scores are multiplied, up to
  // 128 during the softmax).
  float vb[V_HELD ? PER_WAVE : 1][NB][16];
  auto fetch_v = [&](int kc, int nb, float (&v)[16]) {
    const int key0 = kc * 32 + 16 * half;
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const int key = key0 + s;
      v[s] = V[(long long)(key < p.tk ? key : p.tk - 1) * p.sVj + nb * 32 + li];
    }
  };
  // What keys past the end read is put to 0 where V is used, not where it is asked for: a wavefront would wait for it there.
  // (P is 0 there; this keeps an inf or NaN of V out.)
  auto only_keys = [&](int kc, float (&v)[16]) {
    if (kc * 32 + 32 <= p.tk) return;
    const int key0 = kc * 32 + 16 * half;
#pragma unroll
    for (int s = 0; s < 16; s++) v[s] = key0 + s < p.tk ? v[s] : 0.0f;
  };
  auto has = [&](int it) { return wave + ATT_WAVES * it < ncb; };
  auto fetch_held = [&]() {
#pragma unroll
    for (int it = 0; it < (V_HELD ? PER_WAVE : 1); it++)
      if (!SKIP || has(it))
#pragma unroll
        for (int nb = 0; nb < NB; nb++) fetch_v(wave + ATT_WAVES * it, nb, vb[it][nb]);
  };

  // ---- 1. scores -------------------------------------------------------------------
  {
    // Q of the workgroup, then a block of keys for each wavefront: [row][HD + 4 floats]
    constexpr int LP = HD + 4, PPR = HD / 4, KL = 32 * PPR / 64, QL = (32 * PPR + 64 * ATT_WAVES - 1) / (64 * ATT_WAVES);
    constexpr int AHEAD = PER_WAVE < 2 ? PER_WAVE : 2;
    float *const qs = lds, *const ks = lds + (1 + wave) * (32 * LP);
    f32x4 qr[QL], kr[AHEAD][KL];
    const int r0 = lane / PPR, c0 = lane % PPR * 4;
#pragma unroll
    for (int i = 0; i < QL; i++) {
      const int at = tid + i * 64 * ATT_WAVES, row = row0 + at / PPR;
      qr[i] = *reinterpret_cast<const f32x4 *>(Q + (long long)(row < p.tq ? row : p.tq - 1) * p.sQi + at % PPR * 4);  // (rows past the end are never stored)
    }
    auto fetch_k = [&](int it) {
#pragma unroll
      for (int i = 0; i < KL; i++) {
        const int key = (wave + ATT_WAVES * it) * 32 + i * (64 / PPR) + r0;
        kr[it % AHEAD][i] = *reinterpret_cast<const f32x4 *>(K + (long long)(key < p.tk ? key : p.tk - 1) * p.sKj + c0);
      }
    };
#pragma unroll
    for (int it = 0; it < AHEAD; it++)
      if (has(it)) fetch_k(it);
#pragma unroll
    for (int i = 0; i < QL; i++) {
      const int at = tid + i * 64 * ATT_WAVES;
      if (32 * PPR % (64 * ATT_WAVES) == 0 || at < 32 * PPR) *reinterpret_cast<f32x4 *>(qs + at / PPR * LP + at % PPR * 4) = qr[i];
    }
    __syncthreads();
    f32x16 acc[PER_WAVE];
#pragma unroll
    for (int it = 0; it < PER_WAVE; it++) {
      if (!has(it)) break;
#pragma unroll
      for (int i = 0; i < KL; i++) *reinterpret_cast<f32x4 *>(ks + (i * (64 / PPR) + r0) * LP + c0) = kr[it % AHEAD][i];
      if (it + AHEAD < PER_WAVE && has(it + AHEAD)) fetch_k(it + AHEAD);
      if (V_FIRST && it == 0) fetch_held();
      __builtin_amdgcn_wave_barrier();
      acc[it] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < HALF / 4; c++) {
        const f32x4 q = *reinterpret_cast<const f32x4 *>(qs + li * LP + HALF * half + 4 * c);
        const f32x4 k = *reinterpret_cast<const f32x4 *>(ks + li * LP + HALF * half + 4 * c);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[it] = __builtin_amdgcn_mfma_f32_32x32x2f32(q[e], k[e], acc[it], 0, 0, 0);
      }
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();  // the scores go where Q and the keys were
#pragma unroll
    for (int it = 0; it < PER_WAVE; it++) {
      if (!has(it)) break;
      const int key = (wave + ATT_WAVES * it) * 32 + li;
      const bool key_ok = key < p.tk;
      // lane holds column li, rows 8*(r/4) + 4*half + r%4; keys past the end count as -inf
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        lds[row * p.pitch + key] = key_ok ? p.alpha * acc[it][r] : -INFINITY;
      }
    }
  }
  if (V_HELD && !V_FIRST) fetch_held();
  __syncthreads();

  // ---- 2. softmax over each row, in place (softmax.ts:34-57) ------------------------
  // The wavefront's four (two) rows are taken through every step together.
  {
    constexpr int RPW = ATT_ROWS / ATT_WAVES;
    constexpr int PIECES = 32 * ATT_WAVES * PER_WAVE / 256;  // 16-byte pieces per lane
    const int ncols = ncb * 32;  // a multiple of 4
    const float ninf = -INFINITY;
    f32x4 v[RPW][PIECES];
    float mx[RPW], sum[RPW];
#pragma unroll
    for (int j = 0; j < RPW; j++) {
      const float *srow = lds + (wave + ATT_WAVES * j) * p.pitch;
      mx[j] = ninf;
#pragma unroll
      for (int i = 0; i < PIECES; i++) {
        const int c = 4 * lane + 256 * i;
        v[j][i] = c < ncols ? *reinterpret_cast<const f32x4 *>(srow + c) : f32x4{ninf, ninf, ninf, ninf};
#pragma unroll
        for (int e = 0; e < 4; e++) mx[j] = fmaxf(mx[j], v[j][i][e]);  // fmaxf skips NaN, like `if (v > max)`
      }
    }
#pragma unroll
    for (int j = 0; j < RPW; j++) mx[j] = wave_max(mx[j]);
#pragma unroll
    for (int j = 0; j < RPW; j++) {
      sum[j] = 0.0f;
#pragma unroll
      for (int i = 0; i < PIECES; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float ex = 4 * lane + 256 * i + e < p.tk ? exp_f32(v[j][i][e] - mx[j]) : 0.0f;
          v[j][i][e] = ex;
          sum[j] += ex;
        }
    }
#pragma unroll
    for (int j = 0; j < RPW; j++) sum[j] = wave_sum(sum[j]);
#pragma unroll
    for (int j = 0; j < RPW; j++) {
      float *srow = lds + (wave + ATT_WAVES * j) * p.pitch;
      const float inv = 1.0f / sum[j];
#pragma unroll
      for (int i = 0; i < PIECES; i++) {
        const int c = 4 * lane + 256 * i;
        if (c < ncols) {
          f32x4 t;
#pragma unroll
          for (int e = 0; e < 4; e++) t[e] = v[j][i][e] * inv;
          *reinterpret_cast<f32x4 *>(srow + c) = t;
        }
      }
    }
  }
  __syncthreads();

  // ---- 3. output: this wavefront's key blocks -----------------------------------------
  f32x16 o[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
    o[nb] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto fetch_p = [&](int kc, f32x4 (&pa)[4]) {
    const float *prow = lds + li * p.pitch + kc * 32 + 16 * half;
#pragma unroll
    for (int c = 0; c < 4; c++) pa[c] = *reinterpret_cast<const f32x4 *>(prow + 4 * c);
  };
  f32x4 pa[4];
  if constexpr (V_HELD) {
#pragma unroll
    for (int it = 0; it < PER_WAVE; it++) {
      const int kc = wave + ATT_WAVES * it;
      if (kc >= ncb) break;
      fetch_p(kc, pa);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) only_keys(kc, vb[it][nb]);
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int s = 0; s < 16; s++)
          o[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(pa[s >> 2][s & 3], vb[it][nb][s], o[nb], 0, 0, 0);
    }
  } else {
    for (int kc = wave; kc < ncb; kc += ATT_WAVES) {
      fetch_p(kc, pa);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        float vn[16];
        fetch_v(kc, nb, vn);
        only_keys(kc, vn);
#pragma unroll
        for (int s = 0; s < 16; s++)
          o[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(pa[s >> 2][s & 3], vn[s], o[nb], 0, 0, 0);
      }
    }
  }
  __syncthreads();  // every wavefront has read its part of P: the block is free

  // ---- partial blocks added in wavefront order ----------------------------------------
  constexpr int OP = HD + 1;  // row pitch of a partial block
  {
    float *mine = lds + wave * (ATT_ROWS * OP);
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        mine[row * OP + nb * 32 + li] = o[nb][r];
      }
  }
  __syncthreads();
  float *Y = p.Y + (long long)b * p.sYb;
  for (int cell = tid; cell < ATT_ROWS * HD; cell += 64 * ATT_WAVES) {
    const int row = cell / HD, col = cell - row * HD;
    float sum = lds[row * OP + col];
#pragma unroll
    for (int w = 1; w < ATT_WAVES; w++) sum += lds[w * (ATT_ROWS * OP) + row * OP + col];
    if (row0 + row < p.tq) Y[(long long)(row0 + row) * p.sYi + col] = sum;
  }
}

int lds_pitch(int tk) {
  int pitch = (tk + 31) / 32 * 32;
  if ((pitch / 4) % 2 == 0) pitch += 4;  // rows 16 bytes apart modulo the banks: no conflicts in step 3
  return pitch;
}

template <int HD, int ATT_WAVES, int PER_WAVE>
int launch_attention(const AttParams &p, int batch) {
  // Q and a block of keys a wavefront, then the scores block, and later the wavefronts' partial outputs, whichever is larger
  size_t bytes = (size_t)ATT_ROWS * p.pitch * 4;
  const size_t blocks = (size_t)(p.tk + 31) / 32, rows = (size_t)(1 + (blocks < ATT_WAVES ? blocks : ATT_WAVES)) * 32 * (HD + 4) * 4;
  static_assert((1 + ATT_WAVES) * 32 * (HD + 4) * 4 <= 160 * 1024, "LDS");
  if (rows > bytes) bytes = rows;
  const size_t partials = (size_t)ATT_WAVES * ATT_ROWS * (HD + 1) * 4;
  if (partials > bytes) bytes = partials;
  hipLaunchKernelGGL((attention_rows_kernel<HD, ATT_WAVES, PER_WAVE>), dim3((unsigned)((long long)batch * p.row_blocks)),
                     dim3(64 * ATT_WAVES), bytes, wdh::stream(), p);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}
template <int HD>
int launch_attention(const AttParams &p, int batch) {
  // (64: sixteen wavefronts of one block each, 512 keys 18.8 us, eight of two 19.4; 200 keys 11.6 and 11.0)
  if constexpr (HD == 32)
    return p.tk > 512 ? launch_attention<HD, 16, 2>(p, batch) : launch_attention<HD, 16, 1>(p, batch);
  else if constexpr (HD == 64)  // (a launch has at most 2^32 - 1 threads in a direction: twice as many row blocks with eight wavefronts)
    return p.tk <= 256 ? launch_attention<HD, 8, 1>(p, batch)
           : p.tk <= 512 && (long long)batch * p.row_blocks <= 0xffffffffLL / 1024 ? launch_attention<HD, 16, 1>(p, batch)
                                                                                    : launch_attention<HD, 8, 4>(p, batch);
  else
    return p.tk > 256 ? launch_attention<HD, 8, 4>(p, batch) : launch_attention<HD, 8, 1>(p, batch);
}

template <int HD, int ATT_WAVES, int PER_WAVE>
hipError_t allow_lds() {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(attention_rows_kernel<HD, ATT_WAVES, PER_WAVE>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
}

}  // namespace

namespace wdh {
// More than 64 KB of dynamic LDS has to be asked for once per kernel and device (called by
// wdh_init with the device current, so that no launch -- captured ones included -- has to).
int init_attention() {
  for (hipError_t e : {allow_lds<32, 16, 2>(), allow_lds<32, 16, 1>(), allow_lds<64, 8, 4>(), allow_lds<64, 16, 1>(),
                       allow_lds<64, 8, 1>(), allow_lds<128, 8, 4>(), allow_lds<128, 8, 1>()})
    WDH_HIP_CHECK(e);
  return WDH_OK;
}
}  // namespace wdh

using wdh::fail;

extern "C" int wdh_attention(wdh_buf hQ, wdh_buf hK, wdh_buf hV, wdh_buf hY, int batch, int tq,
                             int tk, int d, int64_t sQb, int64_t sQi, int64_t sKb, int64_t sKj,
                             int64_t sVb, int64_t sVj, int64_t sYb, int64_t sYi, float alpha) {
  WDH_REQUIRE_INIT();
  WDH_REQUIRE_COMPUTE_LANE();
  if (batch < 0 || tq < 0 || tk < 0 || d < 0) return fail(WDH_EINVAL, "wdh_attention: negative extent");
  if (d != 32 && d != 64 && d != 128)
    return fail(WDH_EINVAL, "wdh_attention: head dimension %d (32, 64 and 128 are built)", d);
  if (tk > ATT_MAX_KEYS)
    return fail(WDH_EINVAL, "wdh_attention: %d keys (at most %d: a block of scores has to fit in LDS)", tk,
                ATT_MAX_KEYS);
  if (sQb < 0 || sQi < 0 || sKb < 0 || sKj < 0 || sVb < 0 || sVj < 0 || sYb < 0 || sYi < 0)
    return fail(WDH_EINVAL, "wdh_attention: negative stride");
  if (batch == 0 || tq == 0) return WDH_OK;
  if (tk == 0) return fail(WDH_EINVAL, "wdh_attention: no keys");
  if ((sQb | sQi | sKb | sKj) % 4 != 0)
    return fail(WDH_EINVAL, "wdh_attention: strides of Q and K must be multiples of 4 elements");
  const long long row_blocks = (tq + ATT_ROWS - 1) / ATT_ROWS;
  if (batch * row_blocks > 0x7fffffffLL) return fail(WDH_EINVAL, "wdh_attention: too many row blocks");
  auto span = [](long long n0, long long s0, long long n1, long long s1, long long inner) {
    return (n0 - 1) * s0 + (n1 - 1) * s1 + inner;
  };
  void *pq, *pk, *pv, *py;
  if (!wdh::operand(hQ, (size_t)span(batch, sQb, tq, sQi, d) * 4, "wdh_attention: Q", &pq)) return WDH_EINVAL;
  if (!wdh::operand(hK, (size_t)span(batch, sKb, tk, sKj, d) * 4, "wdh_attention: K", &pk)) return WDH_EINVAL;
  if (!wdh::operand(hV, (size_t)span(batch, sVb, tk, sVj, d) * 4, "wdh_attention: V", &pv)) return WDH_EINVAL;
  if (!wdh::operand(hY, (size_t)span(batch, sYb, tq, sYi, d) * 4, "wdh_attention: Y", &py)) return WDH_EINVAL;
  if ((((uintptr_t)pq | (uintptr_t)pk) & 15) != 0)
    return fail(WDH_EINVAL, "wdh_attention: Q and K must be 16-byte aligned");
  if (py == pq || py == pk || py == pv) return fail(WDH_EINVAL, "wdh_attention: Y aliases an input");
  AttParams p;
  p.Q = (const float *)pq; p.K = (const float *)pk; p.V = (const float *)pv; p.Y = (float *)py;
  p.tq = tq; p.tk = tk; p.pitch = lds_pitch(tk); p.row_blocks = (int)row_blocks;
  p.sQb = sQb; p.sQi = sQi; p.sKb = sKb; p.sKj = sKj; p.sVb = sVb; p.sVj = sVj; p.sYb = sYb; p.sYi = sYi;
  p.alpha = alpha;
  if (d == 32) return launch_attention<32>(p, batch);
  if (d == 64) return launch_attention<64>(p, batch);
  return launch_attention<128>(p, batch);
}

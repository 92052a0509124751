// Lays an operand out for half_product.h: strips of 16 rows, scaled row by row, in two f16 parts.
//
// Bound: memory; 4 bytes an element in, 4 out.  A workgroup has four strips, whose wavefronts read the same lines where rows are not
// k-contiguous, and a chunk of K.
#include "half_product.h"

namespace wdhc {

constexpr int PACK_WAVES = 8, PACK_STRIPS = 4;
enum PackSource { PACK_CONTIGUOUS, PACK_STRIDED, PACK_3X3 };

// EXACT: a workgroup has the whole K and scales a row by its largest element (weights that are kept).  Otherwise (a product's
// operand, laid out on every call) it has PACK_CHUNK steps, and a row is scaled by the largest of its first ones, 2^W_ROOM below
// the end of the range; what outgrows that becomes Inf, which the product finds.
template <int SOURCE, bool EXACT>
__global__ __launch_bounds__(PACK_WAVES * 64) void half_pack_kernel(const float *W, HalfOperand out, int rows, int k, long long sr, long long sk) {
  __shared__ unsigned most[PACK_STRIPS][PACK_WAVES / PACK_STRIPS][16], lossy[PACK_STRIPS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, mine = wave % PACK_STRIPS, turn = wave / PACK_STRIPS;
  const int strip = (int)blockIdx.x * PACK_STRIPS + mine, steps = out.steps;
  const int row = strip * 16 + (lane & 15), kk = 8 * (lane >> 4);
  const bool live = strip < out.strips;
  const float *const w = W + (long long)(row < rows ? row : rows - 1) * sr;
  auto load = [&](int step, float (&x)[8]) {
    if (SOURCE == PACK_3X3) {
      // sixteen channels of taps 2 s and 2 s + 1; there is no tenth tap
      const int tap = step % 5 * 2 + (kk >> 4);
      const float *const at = w + (long long)(step / 5 * 16 + (kk & 15)) * 9 + tap;
#pragma unroll
      for (int e = 0; e < 8; e++) x[e] = tap < 9 ? at[e * 9] : 0.0f;
    } else if (SOURCE == PACK_CONTIGUOUS) {
      const int at = step * HSTEP + kk;   // (k % 8 == 0)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const f32x4 v = at < k ? *reinterpret_cast<const f32x4 *>(w + at + 4 * h) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; e++) x[4 * h + e] = v[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int at = step * HSTEP + kk + e;
        x[e] = at < k ? w[at * sk] : 0.0f;
      }
    }
  };
  constexpr int TURNS = PACK_WAVES / PACK_STRIPS;
  unsigned top = 0;
  for (int step = turn; step < (EXACT || steps < PACK_CHUNK ? steps : PACK_CHUNK); step += TURNS) {
    float x[8];
    load(step, x);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const unsigned u = __float_as_uint(x[e]) & 0x7fffffffu;
      top = u > top ? u : top;
    }
  }
#pragma unroll
  for (int d = 16; d < 64; d *= 2) {
    const unsigned u = __shfl_xor(top, d);
    top = u > top ? u : top;
  }
  if (lane < 16) most[mine][turn][lane] = top;
  if (threadIdx.x < PACK_STRIPS) lossy[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TURNS; i++) top = most[mine][i][lane & 15] > top ? most[mine][i][lane & 15] : top;
  const int exponent = scale_exponent(top, EXACT ? W_TARGET : W_TARGET - W_ROOM);
  const float scale = row < rows ? scale_of(exponent) : 0.0f, least = __builtin_ldexpf(1.0f, FULL_EXPONENT - exponent);
  unsigned lost = 0;
  const int first = EXACT ? 0 : (int)blockIdx.y * PACK_CHUNK, end = EXACT || first + PACK_CHUNK > steps ? steps : first + PACK_CHUNK;
  for (int step = first + turn; live && step < end; step += TURNS) {
    float x[8];
    load(step, x);
    const HalfParts q = half_parts(x, scale);
#pragma unroll
    for (int e = 0; e < 8; e++) lost += x[e] != 0.0f && __builtin_fabsf(x[e]) < least ? 1u : 0u;
    unsigned char *const at = out.packed + ((long long)strip * steps + step) * STEP_BYTES + lane * 16;
    *reinterpret_cast<f16x8 *>(at) = q.h;
    *reinterpret_cast<f16x8 *>(at + 1024) = q.l;
  }
  if (lost) atomicAdd(&lossy[mine], lost);
  __syncthreads();
  if (!live || turn > 0) return;
  int *const exps = reinterpret_cast<int *>(out.packed + half_fragment_bytes(out.strips, steps));
  if (lane < 16 && blockIdx.y == 0) exps[row] = exponent;
  if (lane == 0) reinterpret_cast<unsigned *>(exps + out.strips * 16)[strip * out.chunks + (int)blockIdx.y] = lossy[mine];
}

template <int SOURCE, bool EXACT>
static int pack(const float *W, const HalfOperand &out, int rows, int k, long long sr, long long sk) {
  const dim3 grid((unsigned)((out.strips + PACK_STRIPS - 1) / PACK_STRIPS), (unsigned)out.chunks), block(PACK_WAVES * 64);
  hipLaunchKernelGGL((half_pack_kernel<SOURCE, EXACT>), grid, block, 0, wdh::stream(), W, out, rows, k, sr, sk);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}
int half_pack(const float *W, const HalfOperand &out, int rows, int k, long long sr, long long sk) {
  const bool vec = sk == 1 && k % 8 == 0 && sr % 4 == 0 && ((uintptr_t)W & 15) == 0;
  if (out.chunks == 1) return vec ? pack<PACK_CONTIGUOUS, true>(W, out, rows, k, sr, sk) : pack<PACK_STRIDED, true>(W, out, rows, k, sr, sk);
  return vec ? pack<PACK_CONTIGUOUS, false>(W, out, rows, k, sr, sk) : pack<PACK_STRIDED, false>(W, out, rows, k, sr, sk);
}
int half_pack3x3(const float *W, const HalfOperand &out, int cout, int c) { return pack<PACK_3X3, true>(W, out, cout, c * 9, (long long)c * 9, 1); }

}  // namespace wdhc

// Bandwidth-bound elementwise kernels: broadcasting binary ops and unary ops.
//
// Semantics follow the reference CPU operators, which evaluate every element
// in JavaScript double arithmetic and store into the typed output array:
//   Binary7  : src/descriptor_runner/operators/cpu/operators/standard/binary7.ts:16-68,257-291
//   CPUUnary : src/descriptor_runner/operators/cpu/operators/standard/unary.ts:10-32
// For fp32 +,-,*,/ the double-then-round result equals the IEEE fp32 result,
// so those are single fp32 instructions here (compiled with contraction off).
#include <math.h>

#include <type_traits>

#include "common.h"
#include "fastdiv.h"
#include "plane_walk.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int MAXD = 6;

struct BinaryParams {
  const void *L;
  const void *R;
  void *Y;
  long long total;          // number of output elements
  int ndim;                 // after collapsing, >= 1
  unsigned shape[MAXD];     // output shape, outermost first
  long long sl[MAXD];       // element strides of L (0 on broadcast axes)
  long long sr[MAXD];
};

// JavaScript ToInt32 of a double (what storing into an Int32Array does).
__device__ __forceinline__ int js_to_int32(double d) {
  if (!(d == d) || isinf(d)) return 0;
  double t = trunc(d);
  double m = fmod(t, 4294967296.0);
  if (m < 0) m += 4294967296.0;
  return (int)(unsigned)m;
}

template <int OP>
__device__ __forceinline__ float apply_f(float l, float r) {
  if (OP == WDH_BIN_ADD) return l + r;
  if (OP == WDH_BIN_SUB) return l - r;
  if (OP == WDH_BIN_MUL) return l * r;
  if (OP == WDH_BIN_DIV) return l / r;
  // x^2 (a written-out variance): the square of an fp32 number is exact in double, so one fp32 product rounds it
  // the same, and a wavefront whose exponents are all 2 skips pow's few hundred instructions
  // ([8, 95, 126, 192] to the power of a scalar 2: 119.7 -> 31.3 us, 4.6 TB/s)
  if (r == 2.0f) return l * l;
  return (float)pow((double)l, (double)r);
}

// Four at a time, powers with one branch for the four, or none where the caller has asked already (ASK): those of another
// exponent than 2 then run side by side (1 M elements to the power of 3 12.2 us, 14.3 with a branch each and 11.9 with
// none, when squares took pow too).
__device__ __forceinline__ bool all_twos(f32x4 b) { return b.x == 2.0f && b.y == 2.0f && b.z == 2.0f && b.w == 2.0f; }
template <int OP, bool ASK = true>
__device__ __forceinline__ f32x4 apply_f4(f32x4 a, f32x4 b) {
  f32x4 v;
  if (OP == WDH_BIN_POW) {
    if (ASK && all_twos(b)) return a * a;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float y = (float)pow((double)a[e], (double)b[e]);
      v[e] = b[e] == 2.0f ? a[e] * a[e] : y;
    }
    return v;
  }
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = apply_f<OP>(a[e], b[e]);
  return v;
}

// A piece of two or four elements; every element of a piece the same value.
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int UNIT> struct Piece;
template <> struct Piece<2> {
  typedef f32x2 type;
  static __device__ __forceinline__ type same(float s) { return f32x2{s, s}; }
};
template <> struct Piece<4> {
  typedef f32x4 type;
  static __device__ __forceinline__ type same(float s) { return f32x4{s, s, s, s}; }
};
template <int OP, bool ASK = true>
__device__ __forceinline__ f32x4 apply_piece(f32x4 a, f32x4 b) { return apply_f4<OP, ASK>(a, b); }
template <int OP, bool ASK = true>
__device__ __forceinline__ f32x2 apply_piece(f32x2 a, f32x2 b) { return f32x2{apply_f<OP>(a.x, b.x), apply_f<OP>(a.y, b.y)}; }

template <int OP>
__device__ __forceinline__ int apply_i(int l, int r) {
  double a = (double)l, b = (double)r;
  if (OP == WDH_BIN_ADD) return js_to_int32(a + b);
  if (OP == WDH_BIN_SUB) return js_to_int32(a - b);
  if (OP == WDH_BIN_MUL) return js_to_int32(a * b);
  if (OP == WDH_BIN_DIV) return js_to_int32(a / b);
  return js_to_int32(pow(a, b));
}

// Dense fast path: both inputs have the output's shape.  16-byte accesses,
// grid-stride; the tail (total % 4) is handled by the first few threads.
template <int OP>
__global__ __launch_bounds__(256) void binary_dense_f32(const float *__restrict__ L,
                                                        const float *__restrict__ R,
                                                        float *__restrict__ Y,
                                                        long long total) {
  const long long nvec = total >> 2;
  const long long stride = (long long)gridDim.x * blockDim.x;
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const f32x4 *L4 = reinterpret_cast<const f32x4 *>(L);
  const f32x4 *R4 = reinterpret_cast<const f32x4 *>(R);
  f32x4 *Y4 = reinterpret_cast<f32x4 *>(Y);
  for (long long v = i; v < nvec; v += stride) {
    Y4[v] = apply_f4<OP>(L4[v], R4[v]);
  }
  const long long tail = (nvec << 2) + i;
  if (i < (total & 3)) Y[tail] = apply_f<OP>(L[tail], R[tail]);
}

// Broadcast path: the workgroup-tiled walk of plane_walk.h.  UNIT = 4 when the
// innermost axis can be moved in 16-byte pieces: an operand whose innermost
// stride is 1 is read with one 16-byte load, one whose stride is 0 with one
// scalar load.  A thread issues the loads of its four items before it uses any.
template <int OP, typename T, int UNIT>
__global__ __launch_bounds__(256) void binary_plane(BinaryParams p, wdh::PlaneWalk w) {
  const wdh::PlanePos q = wdh::plane_position(w);
  long long bl = 0, br = 0;
#pragma unroll
  for (int d = 0; d < MAXD - 2; d++) {
    if (d < w.nd - 2) {
      bl += (long long)q.oc[d] * p.sl[d];
      br += (long long)q.oc[d] * p.sr[d];
    }
  }
  const unsigned inner = w.shape[w.nd - 1], second = w.shape[w.nd - 2];
  const long long sl2 = p.sl[w.nd - 2], sr2 = p.sr[w.nd - 2];
  const long long sl1 = p.sl[w.nd - 1], sr1 = p.sr[w.nd - 1];
  const T *L = (const T *)p.L, *R = (const T *)p.R;
  T *Y = (T *)p.Y;
  const long long row0 = (long long)q.outer_linear * second;
  if constexpr (UNIT > 1) {
    typedef typename Piece<UNIT>::type V;
    V a[4], b[4];
    bool ok[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const unsigned x = q.x0 + k * q.dx, y = q.y0 + k * q.dy;
      ok[k] = x < inner && y < second;
      if (ok[k]) {
        const float *l = (const float *)L + bl + (long long)y * sl2 + (long long)x * UNIT * sl1;
        const float *r = (const float *)R + br + (long long)y * sr2 + (long long)x * UNIT * sr1;
        if (sl1) a[k] = *reinterpret_cast<const V *>(l);
        else a[k] = Piece<UNIT>::same(*l);
        if (sr1) b[k] = *reinterpret_cast<const V *>(r);
        else b[k] = Piece<UNIT>::same(*r);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (ok[k]) {
        const unsigned x = q.x0 + k * q.dx, y = q.y0 + k * q.dy;
        *reinterpret_cast<V *>((float *)Y + ((row0 + y) * inner + x) * UNIT) = apply_piece<OP>(a[k], b[k]);
      }
    }
  } else {
    T a[4], b[4];
    bool ok[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const unsigned x = q.x0 + k * q.dx, y = q.y0 + k * q.dy;
      ok[k] = x < inner && y < second;
      if (ok[k]) {
        a[k] = L[bl + (long long)y * sl2 + (long long)x * sl1];
        b[k] = R[br + (long long)y * sr2 + (long long)x * sr1];
      }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (ok[k]) {
        const unsigned x = q.x0 + k * q.dx, y = q.y0 + k * q.dy;
        const long long o = (row0 + y) * inner + x;
        if (__is_same(T, float))
          ((float *)Y)[o] = apply_f<OP>((float)a[k], (float)b[k]);
        else
          ((int *)Y)[o] = apply_i<OP>((int)a[k], (int)b[k]);
      }
    }
  }
}

// The flat walk of plane_walk.h over the same views, for rows that fill the tiles above
// badly (a bias added to planes of 56x56 = 784 units): consecutive threads take
// consecutive units of the result whatever the row length.
template <int OP, typename T, int UNIT>
__global__ __launch_bounds__(256) void binary_flat(BinaryParams p, wdh::FlatWalk f, wdh::FastDiv fd_inner) {
  const wdh::FlatPos q = wdh::flat_position(f);
  long long bl = 0, br = 0;
#pragma unroll
  for (int d = 0; d < MAXD - 2; d++) {
    if (d < f.n_outer) {
      bl += (long long)q.oc[d] * p.sl[d];
      br += (long long)q.oc[d] * p.sr[d];
    }
  }
  const int nd = f.n_outer + 2;
  const long long sl2 = p.sl[nd - 2], sr2 = p.sr[nd - 2];
  const long long sl1 = p.sl[nd - 1] * UNIT, sr1 = p.sr[nd - 1] * UNIT;
  const T *L = (const T *)p.L + bl, *R = (const T *)p.R + br;
  T *Y = (T *)p.Y + (long long)q.outer_linear * f.plane * UNIT;
  typedef typename std::conditional<UNIT == 4, f32x4, typename std::conditional<UNIT == 2, f32x2, T>::type>::type V;
  for (unsigned u0 = q.begin + threadIdx.x; u0 < q.end; u0 += 1024) {
    V a[4], b[4];
    bool squares = OP == WDH_BIN_POW && UNIT == 4;  // ([100, 768] to powers of 3 by column: 31.7 us, 33.5 with a branch an item)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const unsigned u = u0 + 256 * k;
      if (u < q.end) {
        const unsigned row = (unsigned)wdh::fdiv((int)u, fd_inner), col = u - row * f.inner;
        const T *l = L + (long long)row * sl2 + (long long)col * sl1;
        const T *r = R + (long long)row * sr2 + (long long)col * sr1;
        if constexpr (UNIT > 1) {
          if (sl1) a[k] = *reinterpret_cast<const V *>(l);
          else a[k] = Piece<UNIT>::same(*l);
          if (sr1) b[k] = *reinterpret_cast<const V *>(r);
          else b[k] = Piece<UNIT>::same(*r);
          if constexpr (UNIT == 4) squares = squares && all_twos(b[k]);
        } else {
          a[k] = *l;
          b[k] = *r;
        }
      }
    }
    auto store = [&](auto value) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const unsigned u = u0 + 256 * k;
        if (u < q.end) *reinterpret_cast<V *>(Y + (long long)u * UNIT) = value(k);
      }
    };
    if constexpr (UNIT == 4) {
      if (squares) store([&](int k) { return a[k] * a[k]; });
      else store([&](int k) { return apply_f4<OP, false>(a[k], b[k]); });
    } else if constexpr (UNIT == 2) {
      store([&](int k) { return apply_piece<OP>(a[k], b[k]); });
    } else if constexpr (__is_same(T, float)) {
      store([&](int k) { return apply_f<OP>(a[k], b[k]); });
    } else {
      store([&](int k) { return apply_i<OP>(a[k], b[k]); });
    }
  }
}

// General path: one output element per thread per step, any strides.
template <int OP, typename T, typename IDX>
__global__ __launch_bounds__(256) void binary_general(BinaryParams p) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const T *L = (const T *)p.L, *R = (const T *)p.R;
  T *Y = (T *)p.Y;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
       i < p.total; i += stride) {
    IDX rem = (IDX)i;
    long long ol = 0, orr = 0;
#pragma unroll
    for (int d = MAXD - 1; d >= 0; d--) {
      if (d < p.ndim) {
        const IDX q = rem / (IDX)p.shape[d];
        const long long c = (long long)(rem - q * (IDX)p.shape[d]);
        rem = q;
        ol += c * p.sl[d];
        orr += c * p.sr[d];
      }
    }
    if (sizeof(T) == 4 && __is_same(T, float))
      ((float *)Y)[i] = apply_f<OP>(((const float *)L)[ol], ((const float *)R)[orr]);
    else
      ((int *)Y)[i] = apply_i<OP>(((const int *)L)[ol], ((const int *)R)[orr]);
  }
}

unsigned grid_for(long long work_items, int per_block) {
  long long blocks = (work_items + per_block - 1) / per_block;
  long long cap = (long long)wdh::compute_units() * 16;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  return (unsigned)blocks;
}

// Shifts the strides of a rank-1 view by the leading axis the walk adds.
BinaryParams for_walk(const BinaryParams &p, const wdh::PlaneWalk &w) {
  if (w.nd == p.ndim) return p;
  BinaryParams s = p;
  for (int d = p.ndim; d > 0; d--) { s.sl[d] = p.sl[d - 1]; s.sr[d] = p.sr[d - 1]; }
  s.sl[0] = s.sr[0] = 0;
  return s;
}

template <int OP>
int launch_binary(const BinaryParams &p, int dtype, bool dense, int unit) {
  hipStream_t st = wdh::stream();
  const bool small = p.total <= 0xffffffffLL;
  wdh::PlaneWalk w;
  wdh::FlatWalk fw;
  if (dtype != 0) unit = 1;
  const unsigned inner_units = p.shape[p.ndim - 1] / (unsigned)unit;
  if (dtype == 0 && dense) {
    hipLaunchKernelGGL(binary_dense_f32<OP>, dim3(grid_for((p.total + 3) / 4, 256)),
                       dim3(256), 0, st, (const float *)p.L, (const float *)p.R,
                       (float *)p.Y, p.total);
  } else if (p.ndim >= 2 &&
             (!wdh::plan_plane_walk(&w, p.ndim, p.shape, inner_units) || wdh::plane_walk_fill(w) < 0.9) &&
             wdh::plan_flat_walk(&fw, p.ndim, p.shape, inner_units)) {
    const dim3 grid(fw.outer * fw.chunks);
    const wdh::FastDiv fd = wdh::make_fastdiv(fw.inner);
    if (unit == 4)
      hipLaunchKernelGGL((binary_flat<OP, float, 4>), grid, dim3(256), 0, st, p, fw, fd);
    else if (unit == 2)
      hipLaunchKernelGGL((binary_flat<OP, float, 2>), grid, dim3(256), 0, st, p, fw, fd);
    else if (dtype == 0)
      hipLaunchKernelGGL((binary_flat<OP, float, 1>), grid, dim3(256), 0, st, p, fw, fd);
    else
      hipLaunchKernelGGL((binary_flat<OP, int, 1>), grid, dim3(256), 0, st, p, fw, fd);
  } else if (unit > 1 && wdh::plan_plane_walk(&w, p.ndim, p.shape, inner_units)) {
    if (unit == 4)
      hipLaunchKernelGGL((binary_plane<OP, float, 4>), wdh::plane_grid(w), dim3(256), 0, st,
                         for_walk(p, w), w);
    else
      hipLaunchKernelGGL((binary_plane<OP, float, 2>), wdh::plane_grid(w), dim3(256), 0, st,
                         for_walk(p, w), w);
  } else if (wdh::plan_plane_walk(&w, p.ndim, p.shape, p.shape[p.ndim - 1])) {
    if (dtype == 0)
      hipLaunchKernelGGL((binary_plane<OP, float, 1>), wdh::plane_grid(w), dim3(256), 0, st,
                         for_walk(p, w), w);
    else
      hipLaunchKernelGGL((binary_plane<OP, int, 1>), wdh::plane_grid(w), dim3(256), 0, st,
                         for_walk(p, w), w);
  } else if (dtype == 0) {
    const dim3 grid(grid_for(p.total, 256));
    if (small)
      hipLaunchKernelGGL((binary_general<OP, float, unsigned>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((binary_general<OP, float, long long>), grid, dim3(256), 0, st, p);
  } else {
    const dim3 grid(grid_for(p.total, 256));
    if (small)
      hipLaunchKernelGGL((binary_general<OP, int, unsigned>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((binary_general<OP, int, long long>), grid, dim3(256), 0, st, p);
  }
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}

// ---- unary ---------------------------------------------------------------

__device__ __forceinline__ float relu_js(float v) {
  // Math.max(v, 0): NaN stays NaN (the comparison is false for it), -0 becomes +0.
  return v <= 0.0f ? 0.0f : v;
}

// (tanh(v/2) + 1) / 2 as the reference writes it, without tanh: with a = e^-|v| it is q = 1 / (1 + a), or a / (1 + a)
// below zero, to a few double ulps, where the sum does not cancel.  Further down the sum's rounding shows in fp32: tanh
// is 2q - 1 rounded to the places it has next to -1, so that adding and taking away the 1 gives the same multiple of
// 2^-53.  Down to -12 that rounding is left out: a double tanh is right to two of those last places, so that the written
// form is off by up to 2^-53 / sigmoid(v), under 2^-35 of the result, and an fp32 result can differ by one ulp where it
// lies that close to a rounding boundary.  One exponential and one division whatever the value ([8, 192, 95, 126]: 94.9 us
// as written; with tanh below -12 only 35.9, but 109 to 118 where such values are among them).
__device__ __forceinline__ double sigmoid_d(double v) {
  const double a = exp(-fabs(v)), q = (v < 0.0 ? a : 1.0) / (1.0 + a);
  return v < -12.0 ? ((2.0 * q - 1.0) + 1.0) / 2.0 : q;
}

template <int OP>
__device__ __forceinline__ float unary_f(float v) {
  if (OP == WDH_UN_RELU) return relu_js(v);
  if (OP == WDH_UN_SIGMOID) return (float)sigmoid_d((double)v);
  if (OP == WDH_UN_SQRT) return (float)sqrt((double)v);
  if (OP == WDH_UN_EXP) return (float)exp((double)v);
  if (OP == WDH_UN_TANH) return (float)tanh((double)v);
  if (OP == WDH_UN_ABS) return fabsf(v);
  if (OP == WDH_UN_NEG) return -v;
  return (float)(1.0 / (double)v);
}

template <int OP>
__global__ __launch_bounds__(256) void unary_f32(const float *__restrict__ X,
                                                 float *__restrict__ Y,
                                                 long long total, bool vec) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (vec) {
    const long long nvec = total >> 2;
    const f32x4 *X4 = reinterpret_cast<const f32x4 *>(X);
    f32x4 *Y4 = reinterpret_cast<f32x4 *>(Y);
    for (long long v = i; v < nvec; v += stride) {
      f32x4 a = X4[v], y;
      y.x = unary_f<OP>(a.x);
      y.y = unary_f<OP>(a.y);
      y.z = unary_f<OP>(a.z);
      y.w = unary_f<OP>(a.w);
      Y4[v] = y;
    }
    const long long tail = (nvec << 2) + i;
    if (i < (total & 3)) Y[tail] = unary_f<OP>(X[tail]);
  } else {
    for (long long e = i; e < total; e += stride) Y[e] = unary_f<OP>(X[e]);
  }
}

__global__ __launch_bounds__(256) void unary_i32(int op, const int *__restrict__ X,
                                                 int *__restrict__ Y, long long total) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += stride) {
    int v = X[e];
    int y;
    if (op == WDH_UN_RELU) y = v > 0 ? v : 0;
    else if (op == WDH_UN_ABS) y = js_to_int32(fabs((double)v));
    else y = js_to_int32(-(double)v);
    Y[e] = y;
  }
}

// Cast between the two data types the runner has: storing a float into an
// Int32Array applies ToInt32, storing an int into a Float32Array rounds to nearest.
__global__ __launch_bounds__(256) void cast_f32_i32(const float *__restrict__ X,
                                                    int *__restrict__ Y, long long total) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride)
    Y[e] = js_to_int32((double)X[e]);
}
__global__ __launch_bounds__(256) void cast_i32_f32(const int *__restrict__ X,
                                                    float *__restrict__ Y, long long total) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride)
    Y[e] = (float)X[e];
}

template <int OP>
int launch_unary(const float *X, float *Y, long long total) {
  bool vec = (((uintptr_t)X | (uintptr_t)Y) & 15) == 0;
  hipLaunchKernelGGL(unary_f32<OP>, dim3(grid_for((total + 3) / 4, 256)), dim3(256),
                     0, wdh::stream(), X, Y, total, vec);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}

}  // namespace

using wdh::fail;

extern "C" int wdh_binary(int op, int dtype, wdh_buf hL, wdh_buf hR, wdh_buf hY,
                          int ndim, const int32_t *out_shape,
                          const int64_t *strides_l, const int64_t *strides_r) {
  WDH_REQUIRE_INIT();
  WDH_REQUIRE_COMPUTE_LANE();
  if (op < WDH_BIN_ADD || op > WDH_BIN_POW)
    return fail(WDH_EINVAL, "wdh_binary: unknown op %d", op);
  if (dtype != 0 && dtype != 1)
    return fail(WDH_EINVAL, "wdh_binary: unknown dtype %d", dtype);
  if (ndim < 0 || ndim > MAXD)
    return fail(WDH_EINVAL, "wdh_binary: ndim %d outside 0..%d", ndim, MAXD);
  if (ndim > 0 && (!out_shape || !strides_l || !strides_r))
    return fail(WDH_EINVAL, "wdh_binary: NULL shape or strides");

  // Collapse: drop extent-1 axes, merge neighbours that are jointly contiguous
  // (or jointly broadcast) in both operands.
  BinaryParams p = {};
  long long total = 1, span_l = 1, span_r = 1;
  int nd = 0;
  for (int d = 0; d < ndim; d++) {
    if (out_shape[d] < 0 || strides_l[d] < 0 || strides_r[d] < 0)
      return fail(WDH_EINVAL, "wdh_binary: negative extent or stride");
    total *= out_shape[d];
    if (out_shape[d] == 1) continue;
    span_l += (long long)(out_shape[d] - 1) * strides_l[d];
    span_r += (long long)(out_shape[d] - 1) * strides_r[d];
    if (nd > 0 && p.sl[nd - 1] == strides_l[d] * out_shape[d] &&
        p.sr[nd - 1] == strides_r[d] * out_shape[d] &&
        (unsigned long long)p.shape[nd - 1] * out_shape[d] <= 0xffffffffULL) {
      p.shape[nd - 1] *= out_shape[d];
      p.sl[nd - 1] = strides_l[d];
      p.sr[nd - 1] = strides_r[d];
    } else {
      p.shape[nd] = out_shape[d];
      p.sl[nd] = strides_l[d];
      p.sr[nd] = strides_r[d];
      nd++;
    }
  }
  if (total == 0) return WDH_OK;
  if (nd == 0) {  // scalar result
    p.shape[0] = 1;
    p.sl[0] = p.sr[0] = 0;
    nd = 1;
  }
  p.ndim = nd;
  p.total = total;
  void *ptr;
  if (!wdh::operand(hL, (size_t)span_l * 4, "wdh_binary: L", &ptr)) return WDH_EINVAL;
  p.L = ptr;
  if (!wdh::operand(hR, (size_t)span_r * 4, "wdh_binary: R", &ptr)) return WDH_EINVAL;
  p.R = ptr;
  if (!wdh::operand(hY, (size_t)total * 4, "wdh_binary: Y", &ptr)) return WDH_EINVAL;
  p.Y = ptr;

  const bool aligned =
      (((uintptr_t)p.L | (uintptr_t)p.R | (uintptr_t)p.Y) & 15) == 0;
  const bool dense = aligned && nd == 1 && p.sl[0] == 1 && p.sr[0] == 1;
  // 16-byte accesses: the output always; an operand that steps by 1 along the
  // innermost axis needs an aligned base and outer strides that are multiples
  // of 4; one that does not step there (stride 0) is read with scalar loads
  auto piece_ok = [&](const void *base, const long long *st, int unit) {
    if (st[nd - 1] == 0) return true;
    if (st[nd - 1] != 1 || ((uintptr_t)base & (4 * unit - 1))) return false;
    for (int d = 0; d + 1 < nd; d++)
      if (st[d] % unit) return false;
    return true;
  };
  // (pieces of two where pieces of four do not fit: a scale by channel over 8 x 192 planes of 95 x 126 29.9 us with single ones, 27.9 with these)
  int unit = 1;
  for (int u : {4, 2})
    if (unit == 1 && ((uintptr_t)p.Y & (4 * u - 1)) == 0 && p.shape[nd - 1] % u == 0 && piece_ok(p.L, p.sl, u) && piece_ok(p.R, p.sr, u))
      unit = u;
  switch (op) {
    case WDH_BIN_ADD: return launch_binary<WDH_BIN_ADD>(p, dtype, dense, unit);
    case WDH_BIN_SUB: return launch_binary<WDH_BIN_SUB>(p, dtype, dense, unit);
    case WDH_BIN_MUL: return launch_binary<WDH_BIN_MUL>(p, dtype, dense, unit);
    case WDH_BIN_DIV: return launch_binary<WDH_BIN_DIV>(p, dtype, dense, unit);
    default: return launch_binary<WDH_BIN_POW>(p, dtype, dense, unit);
  }
}

extern "C" int wdh_unary(int op, int dtype, wdh_buf hX, wdh_buf hY, size_t length) {
  WDH_REQUIRE_INIT();
  WDH_REQUIRE_COMPUTE_LANE();
  if (op < WDH_UN_RELU || op > WDH_UN_RECIPROCAL)
    return fail(WDH_EINVAL, "wdh_unary: unknown op %d", op);
  if (dtype != 0 && dtype != 1)
    return fail(WDH_EINVAL, "wdh_unary: unknown dtype %d", dtype);
  if (dtype == 1 && op != WDH_UN_RELU && op != WDH_UN_ABS && op != WDH_UN_NEG)
    return fail(WDH_EINVAL, "wdh_unary: op %d does not accept int32", op);
  if (length == 0) return WDH_OK;
  void *px, *py;
  if (!wdh::operand(hX, length * 4, "wdh_unary: X", &px)) return WDH_EINVAL;
  if (!wdh::operand(hY, length * 4, "wdh_unary: Y", &py)) return WDH_EINVAL;
  const long long total = (long long)length;
  if (dtype == 1) {
    hipLaunchKernelGGL(unary_i32, dim3(grid_for(total, 256)), dim3(256), 0,
                       wdh::stream(), op, (const int *)px, (int *)py, total);
    WDH_LAUNCH_CHECK();
    return WDH_OK;
  }
  const float *X = (const float *)px;
  float *Y = (float *)py;
  switch (op) {
    case WDH_UN_RELU: return launch_unary<WDH_UN_RELU>(X, Y, total);
    case WDH_UN_SIGMOID: return launch_unary<WDH_UN_SIGMOID>(X, Y, total);
    case WDH_UN_SQRT: return launch_unary<WDH_UN_SQRT>(X, Y, total);
    case WDH_UN_EXP: return launch_unary<WDH_UN_EXP>(X, Y, total);
    case WDH_UN_TANH: return launch_unary<WDH_UN_TANH>(X, Y, total);
    case WDH_UN_ABS: return launch_unary<WDH_UN_ABS>(X, Y, total);
    case WDH_UN_NEG: return launch_unary<WDH_UN_NEG>(X, Y, total);
    default: return launch_unary<WDH_UN_RECIPROCAL>(X, Y, total);
  }
}

extern "C" int wdh_cast(int from_dtype, int to_dtype, wdh_buf hX, wdh_buf hY, size_t length) {
  WDH_REQUIRE_INIT();
  WDH_REQUIRE_COMPUTE_LANE();
  if ((from_dtype != 0 && from_dtype != 1) || (to_dtype != 0 && to_dtype != 1))
    return fail(WDH_EINVAL, "wdh_cast: dtype %d -> %d (0 = float32, 1 = int32)", from_dtype,
                to_dtype);
  if (length == 0) return WDH_OK;
  void *px, *py;
  if (!wdh::operand(hX, length * 4, "wdh_cast: X", &px)) return WDH_EINVAL;
  if (!wdh::operand(hY, length * 4, "wdh_cast: Y", &py)) return WDH_EINVAL;
  const long long total = (long long)length;
  if (from_dtype == to_dtype) {
    WDH_HIP_CHECK(hipMemcpyAsync(py, px, length * 4, hipMemcpyDeviceToDevice, wdh::stream()));
    return WDH_OK;
  }
  if (from_dtype == 0)
    hipLaunchKernelGGL(cast_f32_i32, dim3(grid_for(total, 256)), dim3(256), 0, wdh::stream(),
                       (const float *)px, (int *)py, total);
  else
    hipLaunchKernelGGL(cast_i32_f32, dim3(grid_for(total, 256)), dim3(256), 0, wdh::stream(),
                       (const int *)px, (float *)py, total);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}

// Generic elementwise, broadcast, reduction and strided-copy kernels behind
// the primitive op surface of the engine (ttrl/engine/ops/__init__.py:32-44):
// add/sub/mul/div with tensor, broadcast or scalar operands
// (ttrl/engine/ops/elementwise.py:15-148), the unary ops and their backward
// factors (ttrl/engine/ops/unary.py:21-150), sum/max/argmax along one axis
// (ttrl/engine/ops/reduce.py:12-99), the broadcast-gradient reduction
// (ttrl/engine/ops/broadcast.py:11-54), concat/split/slice copies
// (ttrl/engine/ops/shape.py:10-151) and the device one-hot
// (ttrl/engine/ops/functional.py:112-123).
//
// These serve composed, eager or test-time use of single ops; the hot update
// paths run the fused layer and loss kernels instead.
#include "common.hpp"

#include <cmath>

namespace ttrl {

float* ctx_workspace(ttrl_ctx* ctx, long* floats);  // stream-ordered scratch (runtime.hip)

constexpr int kEwThreads = 256;
constexpr int kMaxDims = 6;

struct Dims {
  int nd;
  long shape[kMaxDims];
  long sa[kMaxDims];
  long sb[kMaxDims];
  long sy[kMaxDims];
};

__device__ inline float unary_op(int op, float x, float s) {
  switch (op) {
    case TTRL_U_RELU: return x > 0.f ? x : 0.f;
    case TTRL_U_ABS: return fabsf(x);
    case TTRL_U_SIGN: return x > 0.f ? 1.f : (x < 0.f ? -1.f : 0.f);
    case TTRL_U_SQUARE: return x * x;
    case TTRL_U_EXP: return expf(x);
    case TTRL_U_LOG: return logf(x);
    case TTRL_U_TANH: return tanhf(x);
    case TTRL_U_SIGMOID: return 1.f / (1.f + expf(-x));
    case TTRL_U_SQRT: return sqrtf(x);
    case TTRL_U_NEG: return -x;
    case TTRL_U_ADD_S: return x + s;
    case TTRL_U_MUL_S: return x * s;
    case TTRL_U_RSUB_S: return s - x;
    case TTRL_U_DIV_S: return x / s;
    case TTRL_U_EQZ: return x == 0.f ? 1.f : 0.f;
    case TTRL_U_GTZ: return x > 0.f ? 1.f : 0.f;
    case TTRL_U_ISFINITE: return isfinite(x) ? 1.f : 0.f;
    default: return x;
  }
}

__device__ inline float binary_op(int op, float a, float b) {
  switch (op) {
    case TTRL_B_ADD: return a + b;
    case TTRL_B_SUB: return a - b;
    case TTRL_B_MUL: return a * b;
    case TTRL_B_DIV: return a / b;
    case TTRL_B_RELU_BW: return b > 0.f ? a : 0.f;
    case TTRL_B_MAX: return fmaxf(a, b);
    case TTRL_B_MIN: return fminf(a, b);
    case TTRL_B_EQ: return a == b ? 1.f : 0.f;
    default: return a;
  }
}

__global__ __launch_bounds__(kEwThreads) void k_unary(int op, const float* __restrict__ a, float* __restrict__ y,
                                                      long n, float s) {
  for (long i = blockIdx.x * long(kEwThreads) + threadIdx.x; i < n; i += long(gridDim.x) * kEwThreads)
    y[i] = unary_op(op, a[i], s);
}

__global__ __launch_bounds__(kEwThreads) void k_binary(int op, const float* __restrict__ a,
                                                       const float* __restrict__ b, float* __restrict__ y, long n,
                                                       Dims d) {
  for (long i = blockIdx.x * long(kEwThreads) + threadIdx.x; i < n; i += long(gridDim.x) * kEwThreads) {
    long rem = i, ia = 0, ib = 0;
    for (int k = d.nd - 1; k >= 0; --k) {
      const long c = rem % d.shape[k];
      rem /= d.shape[k];
      ia += c * d.sa[k];
      ib += c * d.sb[k];
    }
    y[i] = binary_op(op, a[ia], b[ib]);
  }
}

// Operands that are each contiguous or one repeated element (the common
// case): four elements a thread where the pointers are 16-byte aligned, no
// index arithmetic (the general form's 64-bit divisions per axis took 27 us
// for a product of 5.3 M elements, this takes 6.9: HBM's rate).  MA, MB: 1
// contiguous, 0 a scalar.
template <int MA, int MB>
__global__ __launch_bounds__(kEwThreads) void k_binary_flat(int op, const float* __restrict__ a,
                                                            const float* __restrict__ b, float* __restrict__ y, long n,
                                                            int vec) {
  const long first = blockIdx.x * long(kEwThreads) + threadIdx.x, step = long(gridDim.x) * kEwThreads;
  const long nv = vec ? n / 4 : 0;
  const f32x4* a4 = reinterpret_cast<const f32x4*>(a);
  const f32x4* b4 = reinterpret_cast<const f32x4*>(b);
  for (long i = first; i < nv; i += step) {
    const f32x4 u = MA ? a4[i] : f32x4{a[0], a[0], a[0], a[0]};
    const f32x4 v = MB ? b4[i] : f32x4{b[0], b[0], b[0], b[0]};
    f32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = binary_op(op, u[j], v[j]);
    reinterpret_cast<f32x4*>(y)[i] = r;
  }
  for (long i = nv * 4 + first; i < n; i += step) y[i] = binary_op(op, a[MA ? i : 0], b[MB ? i : 0]);
}

__global__ __launch_bounds__(kEwThreads) void k_repeat(const float* __restrict__ a, float* __restrict__ y, long n,
                                                       int vec) {
  const long first = blockIdx.x * long(kEwThreads) + threadIdx.x, step = long(gridDim.x) * kEwThreads;
  const float v = a[0];
  const long nv = vec ? n / 4 : 0;
  for (long i = first; i < nv; i += step) reinterpret_cast<f32x4*>(y)[i] = f32x4{v, v, v, v};
  for (long i = nv * 4 + first; i < n; i += step) y[i] = v;
}

__global__ __launch_bounds__(kEwThreads) void k_copy_strided(const float* __restrict__ a, float* __restrict__ y,
                                                             long n, Dims d) {
  for (long i = blockIdx.x * long(kEwThreads) + threadIdx.x; i < n; i += long(gridDim.x) * kEwThreads) {
    long rem = i, ia = 0, iy = 0;
    for (int k = d.nd - 1; k >= 0; --k) {
      const long c = rem % d.shape[k];
      rem /= d.shape[k];
      ia += c * d.sa[k];
      iy += c * d.sy[k];
    }
    y[iy] = a[ia];
  }
}

// Reduce the middle axis of a [outer][dim][inner] view, one thread per
// output, in index order (deterministic).
__global__ __launch_bounds__(kEwThreads) void k_reduce(int op, const float* __restrict__ a, float* __restrict__ y,
                                                       long outer, long dim, long inner) {
  const long n = outer * inner;
  for (long i = blockIdx.x * long(kEwThreads) + threadIdx.x; i < n; i += long(gridDim.x) * kEwThreads) {
    const long o = i / inner, in = i - o * inner;
    const float* p = a + o * dim * inner + in;
    if (op == TTRL_R_SUM) {
      float s = 0.f;
      for (long k = 0; k < dim; ++k) s += p[k * inner];
      y[i] = s;
    } else if (op == TTRL_R_MAX) {
      float m = p[0];
      for (long k = 1; k < dim; ++k) m = fmaxf(m, p[k * inner]);
      y[i] = m;
    } else {  // argmax, first index of the maximum
      float m = p[0];
      long best = 0;
      for (long k = 1; k < dim; ++k)
        if (p[k * inner] > m) {
          m = p[k * inner];
          best = k;
        }
      y[i] = float(best);
    }
  }
}

// Full sum of a long vector in two launches: workgroup w adds elements
// [w * chunk, (w + 1) * chunk) into part[w] (four independent sums per
// thread, added in a fixed order), then one workgroup adds the parts in
// order.  Bound by HBM once the vector fills the device; one workgroup alone
// waits out a memory round trip per pass of its threads (5.3 M elements with
// scalar loads 4,583 us, with float4 loads 1,322 us, in two launches 5.3 us).
// Up to kSumSingle elements the one workgroup costs less than the second
// launch (16,384: 3.5 against 4.0 us; 32,768: 5.2 against 4.0 us).
constexpr long kSumSingle = 16384;
constexpr int kSumParts = 1024;

// The sum of a[begin, end) by one workgroup: float4 loads where `vec` (a
// 16-byte aligned, begin a multiple of 4), any rest by elements.
__device__ inline float range_sum(const float* __restrict__ a, long begin, long end, bool vec, float* red) {
  f32x4 s{0.f, 0.f, 0.f, 0.f};
  long i = begin + threadIdx.x;
  if (vec) {
    const f32x4* v = reinterpret_cast<const f32x4*>(a);
    for (long q = begin / 4 + threadIdx.x; q < end / 4; q += kEwThreads) s += v[q];
    i = end / 4 * 4 + threadIdx.x;
  }
  for (; i < end; i += kEwThreads) s.x += a[i];
  return block_sum<kEwThreads>((s.x + s.y) + (s.z + s.w), red);
}

__global__ __launch_bounds__(kEwThreads) void k_sum_parts(const float* __restrict__ a, long n, long chunk, int vec,
                                                          float* __restrict__ part) {
  __shared__ float red[kEwThreads / 64];
  const long begin = blockIdx.x * chunk;
  const float t = range_sum(a, begin, begin + chunk < n ? begin + chunk : n, vec != 0, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ __launch_bounds__(kEwThreads) void k_sum_all(const float* __restrict__ a, long n, int vec,
                                                        float* __restrict__ y) {
  __shared__ float red[kEwThreads / 64];
  const float t = range_sum(a, 0, n, vec != 0, red);
  if (threadIdx.x == 0) *y = t;
}

__global__ __launch_bounds__(kEwThreads) void k_onehot(const float* __restrict__ idx, float* __restrict__ y, long B,
                                                       int A) {
  const long n = B * A;
  for (long i = blockIdx.x * long(kEwThreads) + threadIdx.x; i < n; i += long(gridDim.x) * kEwThreads) {
    const long b = i / A;
    const int a = int(i - b * A);
    y[i] = (float(a) - idx[b]) == 0.f ? 1.f : 0.f;
  }
}

inline unsigned ew_grid(long n) {
  long b = (n + kEwThreads - 1) / kEwThreads;
  if (b < 1) b = 1;
  if (b > 4096) b = 4096;
  return unsigned(b);
}

// Which flat form an operand of extents `shape` has: 1 contiguous in index
// order, 0 one element throughout, -1 neither.  Axes of extent 1 do not move
// the operand, so their strides are not read.
int flat_mode(const Dims& d, const long* stride) {
  bool contiguous = true, scalar = true;
  long want = 1;
  for (int k = d.nd - 1; k >= 0; --k) {
    if (d.shape[k] == 1) continue;
    contiguous = contiguous && stride[k] == want;
    scalar = scalar && stride[k] == 0;
    want *= d.shape[k];
  }
  return contiguous ? 1 : scalar ? 0 : -1;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int make_dims(int nd, const long* shape, const long* sa, const long* sb, const long* sy, Dims& d, long& n) {
  TTRL_REQUIRE(nd >= 1 && nd <= kMaxDims, "elementwise: rank %d outside [1, %d]", nd, kMaxDims);
  d.nd = nd;
  n = 1;
  for (int k = 0; k < nd; ++k) {
    TTRL_REQUIRE(shape[k] >= 0, "elementwise: negative extent");
    d.shape[k] = shape[k];
    d.sa[k] = sa ? sa[k] : 0;
    d.sb[k] = sb ? sb[k] : 0;
    d.sy[k] = sy ? sy[k] : 0;
    n *= shape[k];
  }
  return TTRL_OK;
}

}  // namespace ttrl

using namespace ttrl;

extern "C" {

int ttrl_unary(ttrl_ctx* ctx, int op, const float* a, float* y, long n, float scalar) {
  TTRL_REQUIRE(ctx && ((a && y) || n == 0), "ttrl_unary: null argument");
  TTRL_REQUIRE(op >= 0 && op < TTRL_U_COUNT, "ttrl_unary: unknown op %d", op);
  if (n <= 0) return TTRL_OK;
  hipLaunchKernelGGL(k_unary, dim3(ew_grid(n)), dim3(kEwThreads), 0, stream_of(ctx), op, a, y, n, scalar);
  return check_launch("ttrl_unary");
}

int ttrl_binary(ttrl_ctx* ctx, int op, const float* a, const float* b, float* y, int ndim, const long* shape,
                const long* stride_a, const long* stride_b) {
  TTRL_REQUIRE(ctx && a && b && y && shape && stride_a && stride_b, "ttrl_binary: null argument");
  TTRL_REQUIRE(op >= 0 && op < TTRL_B_COUNT, "ttrl_binary: unknown op %d", op);
  Dims d;
  long n = 0;
  int rc = make_dims(ndim, shape, stride_a, stride_b, nullptr, d, n);
  if (rc) return rc;
  if (n <= 0) return TTRL_OK;
  const int ma = flat_mode(d, d.sa), mb = flat_mode(d, d.sb);
  if (ma >= 0 && mb >= 0) {
    const int vec = (!ma || aligned16(a)) && (!mb || aligned16(b)) && aligned16(y);
    const dim3 grid(ew_grid(vec ? (n + 3) / 4 : n)), block(kEwThreads);
    if (ma && mb) hipLaunchKernelGGL((k_binary_flat<1, 1>), grid, block, 0, stream_of(ctx), op, a, b, y, n, vec);
    else if (ma) hipLaunchKernelGGL((k_binary_flat<1, 0>), grid, block, 0, stream_of(ctx), op, a, b, y, n, vec);
    else if (mb) hipLaunchKernelGGL((k_binary_flat<0, 1>), grid, block, 0, stream_of(ctx), op, a, b, y, n, vec);
    else hipLaunchKernelGGL((k_binary_flat<0, 0>), grid, block, 0, stream_of(ctx), op, a, b, y, n, vec);
    return check_launch("ttrl_binary");
  }
  hipLaunchKernelGGL(k_binary, dim3(ew_grid(n)), dim3(kEwThreads), 0, stream_of(ctx), op, a, b, y, n, d);
  return check_launch("ttrl_binary");
}

int ttrl_copy_strided(ttrl_ctx* ctx, const float* a, float* y, int ndim, const long* shape, const long* stride_a,
                      const long* stride_y) {
  TTRL_REQUIRE(ctx && a && y && shape && stride_a && stride_y, "ttrl_copy_strided: null argument");
  Dims d;
  long n = 0;
  int rc = make_dims(ndim, shape, stride_a, nullptr, stride_y, d, n);
  if (rc) return rc;
  if (n <= 0) return TTRL_OK;
  if (flat_mode(d, d.sa) == 0 && flat_mode(d, d.sy) == 1) {  // one element repeated over a dense output
    const int vec = aligned16(y);
    hipLaunchKernelGGL(k_repeat, dim3(ew_grid(vec ? (n + 3) / 4 : n)), dim3(kEwThreads), 0, stream_of(ctx), a, y, n,
                       vec);
    return check_launch("ttrl_copy_strided");
  }
  hipLaunchKernelGGL(k_copy_strided, dim3(ew_grid(n)), dim3(kEwThreads), 0, stream_of(ctx), a, y, n, d);
  return check_launch("ttrl_copy_strided");
}

int ttrl_reduce(ttrl_ctx* ctx, int op, const float* a, float* y, long outer, long dim, long inner) {
  TTRL_REQUIRE(ctx && a && y, "ttrl_reduce: null argument");
  TTRL_REQUIRE(op >= 0 && op < TTRL_R_COUNT, "ttrl_reduce: unknown op %d", op);
  TTRL_REQUIRE(outer >= 1 && dim >= 1 && inner >= 1, "ttrl_reduce: empty extent");
  if (op == TTRL_R_SUM && outer == 1 && inner == 1) {
    const int vec = (reinterpret_cast<uintptr_t>(a) & 15) == 0;
    long wsf = 0;
    float* part = dim > kSumSingle ? ctx_workspace(ctx, &wsf) : nullptr;
    if (part && wsf >= kSumParts) {
      // whole float4s per workgroup, at least one pass of its threads
      long chunk = (dim + kSumParts - 1) / kSumParts;
      chunk = chunk < 4 * kEwThreads ? 4 * kEwThreads : (chunk + 3) / 4 * 4;
      const unsigned blocks = unsigned((dim + chunk - 1) / chunk);
      hipLaunchKernelGGL(k_sum_parts, dim3(blocks), dim3(kEwThreads), 0, stream_of(ctx), a, dim, chunk, vec, part);
      hipLaunchKernelGGL(k_sum_all, dim3(1), dim3(kEwThreads), 0, stream_of(ctx), part, long(blocks), 1, y);
    } else {
      hipLaunchKernelGGL(k_sum_all, dim3(1), dim3(kEwThreads), 0, stream_of(ctx), a, dim, vec, y);
    }
  } else {
    hipLaunchKernelGGL(k_reduce, dim3(ew_grid(outer * inner)), dim3(kEwThreads), 0, stream_of(ctx), op, a, y, outer,
                       dim, inner);
  }
  return check_launch("ttrl_reduce");
}

int ttrl_one_hot(ttrl_ctx* ctx, const float* indices, float* y, long batch, int num_classes) {
  TTRL_REQUIRE(ctx && indices && y, "ttrl_one_hot: null argument");
  TTRL_REQUIRE(batch >= 0 && num_classes > 0, "ttrl_one_hot: bad extents");
  if (batch == 0) return TTRL_OK;
  hipLaunchKernelGGL(k_onehot, dim3(ew_grid(batch * num_classes)), dim3(kEwThreads), 0, stream_of(ctx), indices, y,
                     batch, num_classes);
  return check_launch("ttrl_one_hot");
}

}  // extern "C"

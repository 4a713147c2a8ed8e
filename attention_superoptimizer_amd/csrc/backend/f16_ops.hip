// Kernel-level fp16 operators (the un-fused ops a kernel graph runs outside its
// customized ops).  Arithmetic is fp32 with one fp16 rounding per stored element, the rule
// the reference's generated programs follow (src/kernel/triton_code_gen.cc:246-268).
// Results are row-major; the matmul reads either storage order of its operands (as the
// reference's GEMM call does, src/kernel/cuda/matmul_kernel.cu:61-76), the element-wise
// operators and reductions index their inputs flat, so their callers hand them row-major
// buffers (mi355_f16_transpose makes one from a column-major tensor).  The matmul and the
// transpose are in f16_gemm.hip.
#include "f16_gemm.h"
#include "common.h"

#include <algorithm>

namespace mi355 {

constexpr int kThreads = 256;

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// reference src/kernel/cuda/input_kernel.cu:29-38
__global__ void f16_fill_iota_kernel(_Float16 *x, size_t n, int last_dim) {
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    x[i] = static_cast<_Float16>(static_cast<float>(i % last_dim));
  }
}

__global__ void f16_fill_normal_kernel(_Float16 *x, size_t n, float std, uint64_t seed) {
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    uint64_t r = mix64(seed + i);
    float u1 = (static_cast<float>((r >> 40) & 0xffffff) + 1.0f) * (1.0f / 16777216.0f);
    float u2 = static_cast<float>((r >> 16) & 0xffffff) * (1.0f / 16777216.0f);
    float z = sqrtf(-2.0f * logf(u1)) * cosf(6.28318530717958647692f * u2);
    x[i] = static_cast<_Float16>(z * std);
  }
}

// Element-wise operators move 16 bytes per lane; what is left over (fewer than 8 elements, or
// everything when a base is not 16-byte aligned) goes one element at a time.
__device__ __forceinline__ float f16_binary_value(int op, float x, float y) {
  return (op == KN_ADD_OP) ? x + y : (op == KN_MUL_OP) ? x * y : x / y;
}

__global__ void f16_unary_kernel(int op, _Float16 const *__restrict__ in,
                                 _Float16 *__restrict__ out, size_t n, int vec) {
  size_t const tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  size_t const stride = (size_t)gridDim.x * blockDim.x;
  size_t const n8 = vec ? n / 8 : 0;
  for (size_t i = tid; i < n8; i += stride) {
    half8 v = reinterpret_cast<half8 const *>(in)[i];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      v[j] = static_cast<_Float16>(f16_unary_value(op == KN_EXP_OP, static_cast<float>(v[j])));
    }
    reinterpret_cast<half8 *>(out)[i] = v;
  }
  for (size_t i = n8 * 8 + tid; i < n; i += stride) {
    out[i] = static_cast<_Float16>(f16_unary_value(op == KN_EXP_OP, static_cast<float>(in[i])));
  }
}

struct Dims4 {
  int nd;
  int d1[4], d2[4], od[4];
};

// The reference's broadcast rule, one element per thread (any shapes).
__global__ void f16_binary_kernel(int op, _Float16 const *__restrict__ in1,
                                  _Float16 const *__restrict__ in2, _Float16 *__restrict__ out,
                                  Dims4 D, size_t n) {
  size_t gid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; gid < n; gid += stride) {
    size_t i = gid, s1 = 1, i1 = 0, s2 = 1, i2 = 0;
    for (int d = D.nd - 1; d >= 0; d--) {
      i1 += (i % D.d1[d]) * s1;
      i2 += (i % D.d2[d]) * s2;
      s1 *= D.d1[d];
      s2 *= D.d2[d];
      i /= D.od[d];
    }
    float x = static_cast<float>(in1[i1]), y = static_cast<float>(in2[i2]);
    out[gid] = static_cast<_Float16>(f16_binary_value(op, x, y));
  }
}

// The two shapes that carry the bytes: equal shapes (MODE 0), and a second operand with one
// value per row of the first (last dim 1, MODE 1: the division by row sums); rows are multiples
// of 8 elements, so a lane's eight elements share a row.
template <int MODE>
__global__ void f16_binary_vec_kernel(int op, _Float16 const *__restrict__ in1,
                                      _Float16 const *__restrict__ in2, _Float16 *__restrict__ out,
                                      size_t n8, int row8) {
  size_t const stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n8; i += stride) {
    half8 const a = reinterpret_cast<half8 const *>(in1)[i];
    half8 b;
    if (MODE == 0) {
      b = reinterpret_cast<half8 const *>(in2)[i];
    } else {
      _Float16 const y = in2[i / (size_t)row8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        b[j] = y;
      }
    }
    half8 z;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      z[j] = static_cast<_Float16>(f16_binary_value(op, static_cast<float>(a[j]), static_cast<float>(b[j])));
    }
    reinterpret_cast<half8 *>(out)[i] = z;
  }
}

// Strided sum, the fingerprint kernel's definition (reduction_kernel.cu:86-107): one output per
// thread, `factor` terms `out_stride` apart.  Any shape.
__global__ void f16_reduce_kernel(_Float16 const *__restrict__ in, _Float16 *__restrict__ out,
                                  size_t n_out, int factor, int in_stride, int out_stride) {
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= n_out) {
    return;
  }
  size_t base = (i / out_stride) * (size_t)in_stride + i % out_stride;
  float r = 0.0f;
  for (int k = 0; k < factor; k++) {
    r += static_cast<float>(in[base + (size_t)k * out_stride]);
  }
  out[i] = static_cast<_Float16>(r);
}

// The same with eight neighbouring outputs per thread (out_stride a multiple of 8): every term
// is one 16-byte load and neighbouring threads read neighbouring 16 bytes.
__global__ void f16_reduce_cols_kernel(_Float16 const *__restrict__ in, _Float16 *__restrict__ out,
                                       size_t n_out8, int factor, int in_stride, int out_stride) {
  size_t const i8 = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i8 >= n_out8) {
    return;
  }
  size_t const i = i8 * 8;
  size_t const base = (i / out_stride) * (size_t)in_stride + i % out_stride;
  float r[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int k = 0; k < factor; k++) {
    half8 const v = *reinterpret_cast<half8 const *>(in + base + (size_t)k * out_stride);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      r[j] += static_cast<float>(v[j]);
    }
  }
  half8 o;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    o[j] = static_cast<_Float16>(r[j]);
  }
  *reinterpret_cast<half8 *>(out + i) = o;
}

// Sums of runs of consecutive elements (out_stride 1): 16 lanes per run, 16 bytes per lane and
// step, the lanes' fp32 parts added across the group at the end; runs that are not a multiple
// of 8 elements (or not 16-byte aligned) finish one element at a time.
__global__ void f16_reduce_rows_kernel(_Float16 const *__restrict__ in,
                                       _Float16 *__restrict__ out, size_t n_out, int factor, int vec) {
  int const sub = threadIdx.x % 16;
  size_t const row = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) / 16;
  float r = 0.0f;
  if (row < n_out) {
    _Float16 const *p = in + row * (size_t)factor;
    int const f8 = vec ? factor / 8 : 0;
    for (int k = sub; k < f8; k += 16) {
      half8 const v = reinterpret_cast<half8 const *>(p)[k];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        r += static_cast<float>(v[j]);
      }
    }
    for (int k = f8 * 8 + sub; k < factor; k += 16) {
      r += static_cast<float>(p[k]);
    }
  }
  for (int off = 8; off > 0; off >>= 1) {
    r += __shfl_xor(r, off, 64);
  }
  if (sub == 0 && row < n_out) {
    out[row] = static_cast<_Float16>(r);
  }
}

// eight elements (fewer at the end) of a row of any alignment
__device__ __forceinline__ void store_row_chunk(_Float16 *row, half8 v, int c, int n, bool live) {
  if (live && c + 8 <= n) {
    *reinterpret_cast<half8_any *>(row + c) = v;
  } else if (live) {
#pragma unroll
    for (int u = 0; u < 7; u++) {
      if (c + u < n) {
        row[c + u] = v[u];
      }
    }
  }
}

// exp, row sum and division in one pass: E = exp(X), R = sum of a row of E, P = E / R, each rounded to
// fp16 as the three operators round it (the sum adds the rounded exponentials).  TPR threads own a
// row and keep it in registers, CH chunks of eight elements each, so X is read once and E never:
// two launches and two reads of the score matrix less ([8, 500, 1000]: 16.5 -> 8.7 us; bounded by the
// 24 MB it moves).
template <int TPR, int CH>
__global__ __launch_bounds__(kThreads) void f16_softmax_rows_kernel(_Float16 const *__restrict__ X, _Float16 *__restrict__ E,
                                                                   _Float16 *__restrict__ R, _Float16 *__restrict__ P,
                                                                   size_t rows, int n) {
  size_t const row = blockIdx.x * (size_t)(kThreads / TPR) + threadIdx.x / TPR;
  int const t = threadIdx.x % TPR;
  bool const live = row < rows;
  size_t const at = (live ? row : rows - 1) * (size_t)n;
  half8 v[CH];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < CH; i++) {  // (all loads first)
    int const c = 8 * (i * TPR + t);
    if (c + 8 <= n) {
      v[i] = *reinterpret_cast<half8_any const *>(X + at + c);
    } else {
#pragma unroll
      for (int u = 0; u < 8; u++) {
        v[i][u] = c + u < n ? X[at + c + u] : (_Float16)0.0f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < CH; i++) {
    int const c = 8 * (i * TPR + t);
#pragma unroll
    for (int u = 0; u < 8; u++) {
      v[i][u] = static_cast<_Float16>(f16_unary_value(true, static_cast<float>(v[i][u])));
      sum += c + u < n ? static_cast<float>(v[i][u]) : 0.0f;
    }
    store_row_chunk(E + at, v[i], c, n, live);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
  }
  if (TPR > 64) {
    __shared__ float parts[kThreads / 64];
    parts[threadIdx.x / 64] = sum;
    __syncthreads();
    sum = 0.0f;
#pragma unroll
    for (int w = 0; w < TPR / 64; w++) {
      sum += parts[w];
    }
  }
  _Float16 const total = static_cast<_Float16>(sum);
  if (t == 0 && live) {
    R[row] = total;
  }
#pragma unroll
  for (int i = 0; i < CH; i++) {
    half8 q;
#pragma unroll
    for (int u = 0; u < 8; u++) {
      q[u] = static_cast<_Float16>(static_cast<float>(v[i][u]) / static_cast<float>(total));
    }
    store_row_chunk(P + at, q, 8 * (i * TPR + t), n, live);
  }
}

static inline int grid_for(size_t n) {
  size_t g = (n + kThreads - 1) / kThreads;
  return static_cast<int>(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

}  // namespace mi355

using namespace mi355;

extern "C" int mi355_f16_fill_iota(void *x, size_t n, int last_dim) {
  MI355_REQUIRE_INIT();
  if (last_dim <= 0) {
    return fail(MI355_ERR_INVALID, "last_dim must be positive");
  }
  if (n == 0) {
    return MI355_OK;
  }
  f16_fill_iota_kernel<<<grid_for(n), kThreads, 0, state().stream()>>>(
      static_cast<_Float16 *>(x), n, last_dim);
  MI355_HIP(hipGetLastError());
  return MI355_OK;
}

extern "C" int mi355_f16_fill_normal(void *x, size_t n, float std, uint64_t seed) {
  MI355_REQUIRE_INIT();
  if (n == 0) {
    return MI355_OK;
  }
  f16_fill_normal_kernel<<<grid_for(n), kThreads, 0, state().stream()>>>(
      static_cast<_Float16 *>(x), n, std, seed);
  MI355_HIP(hipGetLastError());
  return MI355_OK;
}

extern "C" int mi355_f16_unary(int op, void const *in, void *out, size_t n) {
  MI355_REQUIRE_INIT();
  if (op != KN_EXP_OP && op != KN_SILU_OP) {
    return fail(MI355_ERR_UNSUPPORTED, "unary op %d", op);
  }
  if (n == 0) {
    return MI355_OK;
  }
  int const vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 ? 1 : 0;
  f16_unary_kernel<<<grid_for(vec ? (n + 7) / 8 : n), kThreads, 0, state().stream()>>>(
      op, static_cast<_Float16 const *>(in), static_cast<_Float16 *>(out), n, vec);
  MI355_HIP(hipGetLastError());
  return MI355_OK;
}

extern "C" int mi355_f16_binary(int op, void const *in1, int const *dims1, void const *in2,
                                int const *dims2, void *out, int const *dims_out,
                                int num_dims) {
  MI355_REQUIRE_INIT();
  if (op != KN_ADD_OP && op != KN_MUL_OP && op != KN_DIV_OP) {
    return fail(MI355_ERR_UNSUPPORTED, "binary op %d", op);
  }
  if (num_dims < 1 || num_dims > 4) {
    return fail(MI355_ERR_INVALID, "num_dims %d out of range", num_dims);
  }
  Dims4 D{};
  D.nd = num_dims;
  size_t n = 1;
  for (int d = 0; d < num_dims; d++) {
    D.d1[d] = dims1[d];
    D.d2[d] = dims2[d];
    D.od[d] = dims_out[d];
    if (dims1[d] <= 0 || dims2[d] <= 0 || dims_out[d] <= 0 ||
        (dims1[d] != dims_out[d] && dims1[d] != 1) ||
        (dims2[d] != dims_out[d] && dims2[d] != 1)) {
      return fail(MI355_ERR_INVALID, "dim %d is not broadcastable", d);
    }
    n *= (size_t)dims_out[d];
  }
  // equal shapes, or one value of the second operand per row of the first: 16 bytes per lane
  bool same = true, row_scalar = num_dims >= 2 && dims2[num_dims - 1] == 1 && dims1[num_dims - 1] == dims_out[num_dims - 1];
  for (int d = 0; d < num_dims; d++) {
    same = same && dims1[d] == dims_out[d] && dims2[d] == dims_out[d];
    if (d < num_dims - 1) {
      row_scalar = row_scalar && dims1[d] == dims_out[d] && dims2[d] == dims_out[d];
    }
  }
  bool const aligned = ((reinterpret_cast<uintptr_t>(in1) | reinterpret_cast<uintptr_t>(out) |
                         (same ? reinterpret_cast<uintptr_t>(in2) : 0)) & 15) == 0;
  int const last = dims_out[num_dims - 1];
  auto const *x1 = static_cast<_Float16 const *>(in1);
  auto const *x2 = static_cast<_Float16 const *>(in2);
  auto *y = static_cast<_Float16 *>(out);
  if (aligned && same && n % 8 == 0) {
    f16_binary_vec_kernel<0><<<grid_for(n / 8), kThreads, 0, state().stream()>>>(op, x1, x2, y, n / 8, 1);
  } else if (aligned && row_scalar && last % 8 == 0 && last > 1) {
    f16_binary_vec_kernel<1><<<grid_for(n / 8), kThreads, 0, state().stream()>>>(op, x1, x2, y, n / 8, last / 8);
  } else {
    f16_binary_kernel<<<grid_for(n), kThreads, 0, state().stream()>>>(op, x1, x2, y, D, n);
  }
  MI355_HIP(hipGetLastError());
  return MI355_OK;
}

extern "C" int mi355_f16_reduce(void const *in, void *out, size_t n_out, int factor,
                                int in_stride, int out_stride) {
  MI355_REQUIRE_INIT();
  if (factor <= 0 || in_stride <= 0 || out_stride <= 0 ||
      (size_t)out_stride * factor != (size_t)in_stride) {
    return fail(MI355_ERR_INVALID, "reduction strides do not match the factor");
  }
  if (n_out == 0) {
    return MI355_OK;
  }
  hipStream_t st = state().stream();
  auto const *x = static_cast<_Float16 const *>(in);
  auto *y = static_cast<_Float16 *>(out);
  bool const aligned = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  if (out_stride == 1 && factor >= 64) {
    int const vec = aligned && factor % 8 == 0 ? 1 : 0;
    size_t const blocks = (n_out * 16 + kThreads - 1) / kThreads;
    f16_reduce_rows_kernel<<<(unsigned)blocks, kThreads, 0, st>>>(x, y, n_out, factor, vec);
  } else if (aligned && out_stride % 8 == 0 && n_out % 8 == 0) {
    size_t const blocks = (n_out / 8 + kThreads - 1) / kThreads;
    f16_reduce_cols_kernel<<<(unsigned)blocks, kThreads, 0, st>>>(x, y, n_out / 8, factor, in_stride, out_stride);
  } else {
    size_t const blocks = (n_out + kThreads - 1) / kThreads;
    f16_reduce_kernel<<<(unsigned)blocks, kThreads, 0, st>>>(x, y, n_out, factor, in_stride, out_stride);
  }
  MI355_HIP(hipGetLastError());
  return MI355_OK;
}

extern "C" int mi355_f16_softmax_rows(void const *X, void *E, void *R, void *P, size_t rows, int n) {
  MI355_REQUIRE_INIT();
  if (n <= 0) {
    return fail(MI355_ERR_INVALID, "row length %d", n);
  }
  if (rows == 0) {
    return MI355_OK;
  }
  auto const *x = static_cast<_Float16 const *>(X);
  auto *e = static_cast<_Float16 *>(E), *r = static_cast<_Float16 *>(R), *p = static_cast<_Float16 *>(P);
  // A wavefront per row while that fills the chip (4 per compute unit) and its registers hold the
  // row, four wavefronts per row otherwise; longer rows one operator after the other.
  bool const wave = rows >= 1024 && n <= 4096;
  int const chunks = (n + 7) / 8, per_thread = (chunks + (wave ? 63 : 255)) / (wave ? 64 : 256);
  size_t const blocks = wave ? (rows + 3) / 4 : rows;
  if (per_thread <= 8 && blocks <= 2147483647u) {
    auto *fn = wave ? (per_thread <= 1   ? f16_softmax_rows_kernel<64, 1>
                       : per_thread <= 2 ? f16_softmax_rows_kernel<64, 2>
                       : per_thread <= 4 ? f16_softmax_rows_kernel<64, 4>
                                         : f16_softmax_rows_kernel<64, 8>)
                    : (per_thread <= 1   ? f16_softmax_rows_kernel<256, 1>
                       : per_thread <= 2 ? f16_softmax_rows_kernel<256, 2>
                                         : f16_softmax_rows_kernel<256, 8>);
    MI355_HIP(launch_kernel(fn, (unsigned)blocks, kThreads, 0, state().stream(), x, e, r, p, rows, n));
    return MI355_OK;
  }
  if (rows > 2147483647u) {
    return fail(MI355_ERR_UNSUPPORTED, "too many rows");
  }
  int const full[2] = {(int)rows, n}, one[2] = {(int)rows, 1};
  if (int rc = mi355_f16_unary(KN_EXP_OP, X, E, rows * (size_t)n)) {
    return rc;
  }
  if (int rc = mi355_f16_reduce(E, R, rows, n, n, 1)) {
    return rc;
  }
  return mi355_f16_binary(KN_DIV_OP, E, full, R, one, P, full, 2);
}

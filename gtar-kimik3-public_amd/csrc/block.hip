// The residual stream and the elementwise parts of the stack's blocks on gfx950, each one pass over memory:
//
//   add_norm    h = residual + y (fp32), x = rmsnorm(h) * weight in bf16: the end of one half block and the start of
//               the next (src/models/kimi_k3.py:39-66 with RMSNorm src/layers/rmsnorm.py:11-16)
//   head_norm   the attention mixer's q and k norms, in place over the heads of a packed q | k | v projection
//   swiglu      silu(gate) * up
//
// All three are bound by HBM.  In PyTorch the stack ran them as 11 to 13 kernels per half block (casts, squares, means,
// products, each a pass of its own): 9.5 ms of the 23.4 ms forward at 72,292 tokens, hidden 1024, against 2.4 ms here.
// Sums and products are fp32 and every result is rounded once.
#include "gdr_common.h"
#include "gdr_internal.h"

namespace gdr {
namespace {

constexpr int kThreads = 256;
constexpr int kRowsPerBlock = kThreads / kWave;
static_assert(kRowsPerBlock == kAddNormRows && kThreads / 16 == kHeadNormRows, "row limits of the entry points");

using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
using f32x4 = float __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
  const f32x4 a = reinterpret_cast<const f32x4*>(p)[0], b = reinterpret_cast<const f32x4*>(p)[1];
#pragma unroll
  for (int i = 0; i < 4; ++i) { x[i] = a[i]; x[4 + i] = b[i]; }
}
__device__ __forceinline__ void load8(const __bf16* p, float (&x)[8]) {
  const bf16x8 a = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = static_cast<float>(a[i]);
}
__device__ __forceinline__ void store8(float* p, const float (&x)[8]) {
  reinterpret_cast<f32x4*>(p)[0] = f32x4{x[0], x[1], x[2], x[3]};
  reinterpret_cast<f32x4*>(p)[1] = f32x4{x[4], x[5], x[6], x[7]};
}
__device__ __forceinline__ void store8(__bf16* p, const float (&x)[8]) {
  bf16x8 a;
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = static_cast<__bf16>(x[i]);
  *reinterpret_cast<bf16x8*>(p) = a;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int m = 1; m < kWave; m *= 2) x = xor_sum(x, m);
  return x;
}

// One wave per row, the row in registers (8 kIt values per lane), so each operand crosses HBM once and a block needs no
// barrier: 72,292 rows of 1,024 (fp32 residual in and out, bf16 addend in, bf16 out: 888 MB).  sum may be the residual
// (each element is read and written by one lane), so neither is restrict.
template <typename RT, int kIt>
__global__ __launch_bounds__(kThreads) void add_norm_kernel(const gdr_add_norm_args a) {
  const int lane = threadIdx.x % kWave;
  const int64_t row = int64_t(blockIdx.x) * kRowsPerBlock + threadIdx.x / kWave;
  if (row >= a.rows) return;
  const RT* res = static_cast<const RT*>(a.residual) + row * a.dim;
  const __bf16* add = a.add ? static_cast<const __bf16*>(a.add) + row * a.dim : nullptr;
  float x[kIt][8];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int c = (it * kWave + lane) * 8;
    if (c < a.dim) {
      load8(res + c, x[it]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[it][i] = 0.f;
    }
  }
  if (add) {
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
      const int c = (it * kWave + lane) * 8;
      if (c < a.dim) {
        float y[8];
        load8(add + c, y);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[it][i] += y[i];
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int c = (it * kWave + lane) * 8;
    if (a.sum && c < a.dim) store8(a.sum + row * a.dim + c, x[it]);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(x[it][i], x[it][i], ss);
  }
  if (!a.out) return;
  const float r = rsqrtf(wave_sum(ss) / float(a.dim) + a.eps);
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int c = (it * kWave + lane) * 8;
    if (c < a.dim) {
      float w[8];
      load8(a.weight + c, w);
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] *= x[it][i] * r;
      store8(static_cast<__bf16*>(a.out) + row * a.dim + c, w);
    }
  }
}

// Any row length and alignment: one value at a time, the sum recomputed for the second pass over the row.
template <typename RT>
__global__ __launch_bounds__(kThreads) void add_norm_any_kernel(const gdr_add_norm_args a) {
  const int lane = threadIdx.x % kWave;
  const int64_t row = int64_t(blockIdx.x) * kRowsPerBlock + threadIdx.x / kWave;
  if (row >= a.rows) return;
  const RT* res = static_cast<const RT*>(a.residual) + row * a.dim;
  const __bf16* add = a.add ? static_cast<const __bf16*>(a.add) + row * a.dim : nullptr;
  auto value = [&](int c) { return static_cast<float>(res[c]) + (add ? static_cast<float>(add[c]) : 0.f); };
  float ss = 0.f;
  for (int c = lane; c < a.dim; c += kWave) ss = __builtin_fmaf(value(c), value(c), ss);
  const float r = a.out ? rsqrtf(wave_sum(ss) / float(a.dim) + a.eps) : 0.f;
  for (int c = lane; c < a.dim; c += kWave) {
    const float x = value(c);
    if (a.sum) a.sum[row * a.dim + c] = x;
    if (a.out) static_cast<__bf16*>(a.out)[row * a.dim + c] = static_cast<__bf16>(a.weight[c] * (x * r));
  }
}

template <typename RT>
hipError_t launch_add_norm_t(const gdr_add_norm_args& a, hipStream_t stream) {
  const dim3 grid(unsigned((a.rows + kRowsPerBlock - 1) / kRowsPerBlock)), block(kThreads);
  const uintptr_t bits = reinterpret_cast<uintptr_t>(a.residual) | reinterpret_cast<uintptr_t>(a.add) |
                         reinterpret_cast<uintptr_t>(a.weight) | reinterpret_cast<uintptr_t>(a.sum) |
                         reinterpret_cast<uintptr_t>(a.out);
  // 16-byte rows of up to 4,096 values stay in registers.
  const int it = a.dim % 8 == 0 && bits % 16 == 0 ? (a.dim + 511) / 512 : 9;
  if (it <= 1) hipLaunchKernelGGL((add_norm_kernel<RT, 1>), grid, block, 0, stream, a);
  else if (it <= 2) hipLaunchKernelGGL((add_norm_kernel<RT, 2>), grid, block, 0, stream, a);
  else if (it <= 4) hipLaunchKernelGGL((add_norm_kernel<RT, 4>), grid, block, 0, stream, a);
  else if (it <= 8) hipLaunchKernelGGL((add_norm_kernel<RT, 8>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((add_norm_any_kernel<RT>), grid, block, 0, stream, a);
  return hipGetLastError();
}

// Sixteen lanes per (token, head) row of 64 or 128 values, rows 0..q_heads-1 of a token with q_weight, the k_heads
// after them with k_weight; the rows are rewritten where they are.
template <int kPer>  // values per lane: 4 or 8
__global__ __launch_bounds__(kThreads) void head_norm_kernel(const gdr_head_norm_args a) {
  constexpr int kDim = 16 * kPer;
  using Vec = __bf16 __attribute__((ext_vector_type(kPer)));
  const int heads = a.q_heads + a.k_heads;
  const int64_t row = int64_t(blockIdx.x) * (kThreads / 16) + threadIdx.x / 16;
  if (row >= a.tokens * heads) return;  // whole 16-lane rows leave together
  const int sub = threadIdx.x % 16, h = int(row % heads);
  Vec* p = reinterpret_cast<Vec*>(static_cast<__bf16*>(a.x) + (row / heads) * a.stride_t + h * kDim + sub * kPer);
  const Vec v = *p;
  const float* w = (h < a.q_heads ? a.q_weight : a.k_weight) + sub * kPer;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) ss += static_cast<float>(v[i]) * static_cast<float>(v[i]);
#pragma unroll
  for (int m = 1; m < 16; m *= 2) ss = xor_sum(ss, m);
  const float r = rsqrtf(ss / float(kDim) + a.eps);
  Vec o;
#pragma unroll
  for (int i = 0; i < kPer; ++i) o[i] = static_cast<__bf16>(w[i] * (static_cast<float>(v[i]) * r));
  *p = o;
}

template <int kVec>  // 8 (16-byte rows) or 1
__global__ __launch_bounds__(kThreads) void swiglu_kernel(const gdr_swiglu_args a) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const uint32_t per_row = uint32_t(a.dim / kVec);
  if (i >= a.rows * per_row) return;
  const int64_t row = i / per_row;
  const int c = int(i - row * per_row) * kVec;
  const __bf16* g = static_cast<const __bf16*>(a.gate) + row * a.stride + c;
  const __bf16* u = static_cast<const __bf16*>(a.up) + row * a.stride + c;
  __bf16* o = static_cast<__bf16*>(a.out) + row * a.dim + c;
  if constexpr (kVec == 8) {
    float x[8], y[8];
    load8(g, x);
    load8(u, y);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = silu_rcp(x[k]) * y[k];
    store8(o, x);
  } else {
    *o = static_cast<__bf16>(silu_rcp(static_cast<float>(*g)) * static_cast<float>(*u));
  }
}

}  // namespace

hipError_t launch_add_norm(const gdr_add_norm_args& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  return a.residual_dtype == GDR_F32 ? launch_add_norm_t<float>(a, stream) : launch_add_norm_t<__bf16>(a, stream);
}

hipError_t launch_head_norm(const gdr_head_norm_args& a, hipStream_t stream) {
  const int64_t rows = a.tokens * (a.q_heads + a.k_heads);
  if (rows == 0) return hipSuccess;
  const dim3 grid(unsigned((rows + kThreads / 16 - 1) / (kThreads / 16)));
  if (a.head_dim == 64) hipLaunchKernelGGL((head_norm_kernel<4>), grid, dim3(kThreads), 0, stream, a);
  else hipLaunchKernelGGL((head_norm_kernel<8>), grid, dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_swiglu(const gdr_swiglu_args& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  const bool wide = swiglu_wide(a);
  const int64_t n = a.rows * (wide ? a.dim / 8 : a.dim);
  const dim3 grid(unsigned((n + kThreads - 1) / kThreads));
  if (wide) hipLaunchKernelGGL((swiglu_kernel<8>), grid, dim3(kThreads), 0, stream, a);
  else hipLaunchKernelGGL((swiglu_kernel<1>), grid, dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace gdr

// Row-wise neighbours of a multi-row layer (prompt prefill, speculative
// verify) around the library matrix products, one launch each:
//   add_rmsnorm  x = x + y (the residual sum), h = _rmsnorm(x, w)
//   add_parts_rmsnorm  the same with y as fp32 shares of a product split over k
//   swiglu_rows  act = silu(gate) * up over the two halves of a gate_up row
//
// Follows src/solort/model/cuda_graph_executor.py:25-28 (_rmsnorm), :131-135
// and :264-267 with the rounding of its bf16 tensors: the residual sum, the
// normalised row, silu(gate) and the product each rounded once, the norm in
// fp32.
//
// Bound: HBM / launch latency.  As torch ops a norm is eight launches over
// fp32 copies of the row (convert, square, mean, add, rsqrt, two products with
// the weight's conversion, convert) and the SwiGLU two.  Measured on MI355X,
// Qwen3-4B widths, per layer with everything else unchanged: 58 us less at 128
// prompt rows (prefill of 8 layers 1796 -> 1332 us), 104 us less at 1024 rows
// (4 layers 1795 -> 1380 us), 55 us less at 5 verify rows (8 layers 1561 ->
// 1125 us).
#include "common.h"
#include "capi_internal.h"

namespace solort {

// Rounded to bf16 the same as with expf, for each of the 65281 bf16 gates that are no NaN (compared one by one).
__device__ __forceinline__ float silu_bf16_rows(float g) { return rbf(g / (1.0f + __expf(-g))); }

// One 256-thread workgroup per row; a thread keeps its first kNormReg 16-byte
// chunks in registers (k <= 8192 in one read), longer rows re-read the rest
// (after ADD from x_out, which the same thread wrote).
constexpr int kNormReg = 4;

template <bool ADD>
__device__ __forceinline__ uint4 add_chunk(const uint16_t* x, const uint16_t* y, uint16_t* x_out, int i) {
  uint4 c = *reinterpret_cast<const uint4*>(x + 8 * i);
  if constexpr (ADD) {
    float a[8], b[8];
    unpack8(c, a);
    unpack8(*reinterpret_cast<const uint4*>(y + 8 * i), b);
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] += b[e];
    c = pack8(a);
    *reinterpret_cast<uint4*>(x_out + 8 * i) = c;
  }
  return c;
}

template <bool ADD>
__global__ __launch_bounds__(256) void add_rmsnorm_kernel(const uint16_t* x, int64_t x_stride, const uint16_t* y,
                                                          int64_t y_stride, const uint16_t* __restrict__ w, int k,
                                                          float eps, uint16_t* x_out, int64_t xo_stride,
                                                          uint16_t* __restrict__ h, int64_t h_stride) {
  __shared__ float s_red[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, nch = k >> 3;
  x += row * x_stride;
  h += row * h_stride;
  if constexpr (ADD) {
    y += row * y_stride;
    x_out += row * xo_stride;
  }
  uint4 c[kNormReg], g[kNormReg];
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < kNormReg; ++q) {
    const int i = tid + 256 * q;
    if (i < nch) {
      g[q] = *reinterpret_cast<const uint4*>(w + 8 * i);
      c[q] = add_chunk<ADD>(x, y, x_out, i);
      float v[8];
      unpack8(c[q], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    }
  }
  for (int i = tid + 256 * kNormReg; i < nch; i += 256) {
    float v[8];
    unpack8(add_chunk<ADD>(x, y, x_out, i), v);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) s_red[tid >> 6] = ss;
  __syncthreads();
  const float r = 1.0f / __builtin_sqrtf((s_red[0] + s_red[1] + s_red[2] + s_red[3]) / (float)k + eps);
#pragma unroll
  for (int q = 0; q < kNormReg; ++q) {
    const int i = tid + 256 * q;
    if (i < nch) {
      float v[8], gv[8];
      unpack8(c[q], v);
      unpack8(g[q], gv);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (v[e] * r) * gv[e];
      *reinterpret_cast<uint4*>(h + 8 * i) = pack8(v);
    }
  }
  const uint16_t* again = ADD ? x_out : x;
  for (int i = tid + 256 * kNormReg; i < nch; i += 256) {
    float v[8], gv[8];
    unpack8(*reinterpret_cast<const uint4*>(again + 8 * i), v);
    unpack8(*reinterpret_cast<const uint4*>(w + 8 * i), gv);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (v[e] * r) * gv[e];
    *reinterpret_cast<uint4*>(h + 8 * i) = pack8(v);
  }
}

// x_out = x + bf16(sum of the n_parts fp32 shares of y), h = _rmsnorm(x_out, w) (NORM): the end of a product whose
// k was split over workgroups (solort_gemm_tile).  One workgroup per row, a thread per 16-byte chunk of the row (two
// above k = 4096), so that a row's shares are all in flight at once; the shares are added in order.
template <bool NORM>
__global__ __launch_bounds__(512) void add_parts_rmsnorm_kernel(const uint16_t* x, int64_t x_stride,
                                                                const float* __restrict__ parts, int n_parts,
                                                                const uint16_t* __restrict__ w, int m, int k, float eps,
                                                                uint16_t* x_out, int64_t xo_stride,
                                                                uint16_t* __restrict__ h, int64_t h_stride) {
  __shared__ float s_red[8];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, nch = k >> 3, nw = blockDim.x >> 6;
  const float* p = parts + row * k;
  const int64_t part = (int64_t)m * k;
  float v[2][8];
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = tid + (int)blockDim.x * q;
    if (i >= nch) break;
    float y[8] = {};
#pragma unroll 4
    for (int s = 0; s < n_parts; ++s) {
      const float4 a = *reinterpret_cast<const float4*>(p + s * part + 8 * i);
      const float4 b = *reinterpret_cast<const float4*>(p + s * part + 8 * i + 4);
      y[0] += a.x; y[1] += a.y; y[2] += a.z; y[3] += a.w;
      y[4] += b.x; y[5] += b.y; y[6] += b.z; y[7] += b.w;
    }
    unpack8(*reinterpret_cast<const uint4*>(x + row * x_stride + 8 * i), v[q]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[q][e] += rbf(y[e]);
    const uint4 c = pack8(v[q]);
    *reinterpret_cast<uint4*>(x_out + row * xo_stride + 8 * i) = c;
    if constexpr (NORM) {
      unpack8(c, v[q]);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[q][e], v[q][e], ss);
    }
  }
  if constexpr (NORM) {
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_red[tid >> 6] = ss;
    __syncthreads();
    float total = 0.f;
    for (int i = 0; i < nw; ++i) total += s_red[i];
    const float r = 1.0f / __builtin_sqrtf(total / (float)k + eps);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = tid + (int)blockDim.x * q;
      if (i >= nch) break;
      float gv[8];
      unpack8(*reinterpret_cast<const uint4*>(w + 8 * i), gv);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[q][e] = (v[q][e] * r) * gv[e];
      *reinterpret_cast<uint4*>(h + row * h_stride + 8 * i) = pack8(v[q]);
    }
  }
}

// One 16-byte chunk of the output per thread.
__global__ __launch_bounds__(256) void swiglu_rows_kernel(const uint16_t* __restrict__ gu, int64_t gu_stride, int m,
                                                          int inter, uint16_t* __restrict__ out, int64_t out_stride) {
  const int nch = inter >> 3, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= nch) return;
  const int64_t row = blockIdx.y;
  const uint16_t* p = gu + row * gu_stride + 8 * c;
  float g[8], u[8];
  unpack8(*reinterpret_cast<const uint4*>(p), g);
  unpack8(*reinterpret_cast<const uint4*>(p + inter), u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = silu_bf16_rows(g[e]) * u[e];
  *reinterpret_cast<uint4*>(out + row * out_stride + 8 * c) = pack8(g);
}

}  // namespace solort

using namespace solort;

extern "C" int solort_add_rmsnorm(const void* x, int64_t x_row_stride, const void* y, int64_t y_row_stride,
                                  const void* norm_w, float eps, int m, int k, void* x_out, int64_t x_out_row_stride,
                                  void* h, int64_t h_row_stride, solort_stream_t stream) {
  const char* name = "add_rmsnorm";
  if (!x || !norm_w || !h || (y && !x_out)) return set_error(SOLORT_EINVAL, "%s: null pointer", name);
  if (m < 1 || k < 8 || k % 8 != 0 || k > 65536)
    return set_error(SOLORT_EINVAL, "%s: bad shape m=%d k=%d (k a multiple of 8, <= 65536)", name, m, k);
  if (x_row_stride < k || h_row_stride < k || (y && (y_row_stride < k || x_out_row_stride < k)) ||
      x_row_stride % 8 || h_row_stride % 8 || (y && (y_row_stride % 8 || x_out_row_stride % 8)))
    return set_error(SOLORT_EINVAL, "%s: row strides must be multiples of 8, at least k", name);
  if (!aligned16(x) || !aligned16(norm_w) || !aligned16(h) || (y && (!aligned16(y) || !aligned16(x_out))))
    return set_error(SOLORT_EINVAL, "%s: pointers must be 16-byte aligned", name);
  if (y)
    hipLaunchKernelGGL(add_rmsnorm_kernel<true>, dim3(m), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x,
                       x_row_stride, (const uint16_t*)y, y_row_stride, (const uint16_t*)norm_w, k, eps,
                       (uint16_t*)x_out, x_out_row_stride, (uint16_t*)h, h_row_stride);
  else
    hipLaunchKernelGGL(add_rmsnorm_kernel<false>, dim3(m), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x,
                       x_row_stride, nullptr, (int64_t)0, (const uint16_t*)norm_w, k, eps, nullptr, (int64_t)0,
                       (uint16_t*)h, h_row_stride);
  return check_launch(name);
}

extern "C" int solort_add_parts_rmsnorm(const void* x, int64_t x_row_stride, const void* parts, int n_parts,
                                        const void* norm_w, float eps, int m, int k, void* x_out,
                                        int64_t x_out_row_stride, void* h, int64_t h_row_stride,
                                        solort_stream_t stream) {
  const char* name = "add_parts_rmsnorm";
  if (!x || !parts || !x_out || (norm_w && !h)) return set_error(SOLORT_EINVAL, "%s: null pointer", name);
  if (m < 1 || k < 8 || k % 8 != 0 || k > 8192 || n_parts < 1)
    return set_error(SOLORT_EINVAL, "%s: bad shape m=%d k=%d n_parts=%d (k a multiple of 8, <= 8192)", name, m, k,
                     n_parts);
  if (x_row_stride < k || x_out_row_stride < k || (norm_w && h_row_stride < k) || x_row_stride % 8 ||
      x_out_row_stride % 8 || (norm_w && h_row_stride % 8))
    return set_error(SOLORT_EINVAL, "%s: row strides must be multiples of 8, at least k", name);
  if (!aligned16(x) || !aligned16(parts) || !aligned16(x_out) || (norm_w && (!aligned16(norm_w) || !aligned16(h))))
    return set_error(SOLORT_EINVAL, "%s: pointers must be 16-byte aligned", name);
  const int nch = k / 8, per = (nch + 511) / 512, threads = ((nch + per - 1) / per + 63) / 64 * 64;
  if (norm_w)
    hipLaunchKernelGGL(add_parts_rmsnorm_kernel<true>, dim3(m), dim3(threads), 0, (hipStream_t)stream,
                       (const uint16_t*)x, x_row_stride, (const float*)parts, n_parts, (const uint16_t*)norm_w, m, k,
                       eps, (uint16_t*)x_out, x_out_row_stride, (uint16_t*)h, h_row_stride);
  else
    hipLaunchKernelGGL(add_parts_rmsnorm_kernel<false>, dim3(m), dim3(threads), 0, (hipStream_t)stream,
                       (const uint16_t*)x, x_row_stride, (const float*)parts, n_parts, nullptr, m, k, eps,
                       (uint16_t*)x_out, x_out_row_stride, nullptr, (int64_t)0);
  return check_launch(name);
}

extern "C" int solort_swiglu_rows(const void* gu, int64_t gu_row_stride, int m, int inter, void* out,
                                  int64_t out_row_stride, solort_stream_t stream) {
  const char* name = "swiglu_rows";
  if (!gu || !out) return set_error(SOLORT_EINVAL, "%s: null pointer", name);
  if (m < 1 || m > 65535 || inter < 8 || inter % 8 != 0 || inter > (1 << 28))
    return set_error(SOLORT_EINVAL, "%s: bad shape m=%d inter=%d (m <= 65535, inter a multiple of 8)", name, m, inter);
  if (gu_row_stride < 2 * (int64_t)inter || out_row_stride < inter || gu_row_stride % 8 || out_row_stride % 8)
    return set_error(SOLORT_EINVAL, "%s: bad row stride", name);
  if (!aligned16(gu) || !aligned16(out)) return set_error(SOLORT_EINVAL, "%s: pointers must be 16-byte aligned", name);
  hipLaunchKernelGGL(swiglu_rows_kernel, dim3((inter / 8 + 255) / 256, m), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)gu, gu_row_stride, m, inter, (uint16_t*)out, out_row_stride);
  return check_launch(name);
}

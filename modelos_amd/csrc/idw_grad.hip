// Elementwise ends of the distance (idw) scores' gradients, float32, gfx950.
//
// The products themselves are batched GEMMs over the 2 heads (head, half)
// blocks; what is left around them are row sums of squares (|q|^2, |k|^2 of
// the distances) and out = 2 (P - x s), P a product [batches, rows, dim], x the
// queries or keys, s a factor per row (sums of the distance coefficients).
// Bound by memory: each operand once. Queries are read, and their gradient
// written, in their own [rows, batches, dim] layout, so no transposed copy is
// made. Against torch's mul, sub, mul and transposing copy (4096 tokens x 4
// heads x 256): 27 -> 9 us; the square and its sum 15 -> 5 us.
// The roundings are the op sequence's: no contraction in the finish.
#include "pkm_common.h"

namespace pkm {

// element offset of row t of batch b
__device__ __forceinline__ int64_t idw_row(int64_t b, int64_t t, int64_t B, int64_t T, int dim, int row_major) {
  return (row_major ? t * B + b : b * T + t) * dim;
}

#pragma clang fp contract(off)
__global__ __launch_bounds__(256) void idw_finish_kernel(const float* __restrict__ P, const float* __restrict__ x,
                                                         const float* __restrict__ s, int64_t B, int64_t T, int dim,
                                                         int row_major, float* __restrict__ out) {
  const int per = dim / 4;
  const int64_t n = B * T * per;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / per;  // in the order of x and out
    const int c = (int)(i - row * per) * 4;
    const int64_t b = row_major ? row % B : row / T, t = row_major ? row / B : row % T;
    const float4 p = *(const float4*)(P + (b * T + t) * dim + c);
    const float4 v = *(const float4*)(x + row * dim + c);
    const float f = s[b * T + t];
    float4 o;
    o.x = 2.f * (p.x - v.x * f);
    o.y = 2.f * (p.y - v.y * f);
    o.z = 2.f * (p.z - v.z * f);
    o.w = 2.f * (p.w - v.w * f);
    *(float4*)(out + row * dim + c) = o;
  }
}
#pragma clang fp contract(on)

// 16 lanes a row, the grid's workgroups over all rows.
__global__ __launch_bounds__(256) void row_sumsq_kernel(const float* __restrict__ x, int64_t B, int64_t T, int dim,
                                                        int row_major, float* __restrict__ out) {
  const int gl = threadIdx.x & 15;
  for (int64_t i = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4); i < B * T; i += (int64_t)gridDim.x * 16) {
    const int64_t b = i / T, t = i - b * T;
    const float* row = x + idw_row(b, t, B, T, dim, row_major);
    float a = 0.f;
    for (int c = 4 * gl; c < dim; c += 64) {
      const float4 v = *(const float4*)(row + c);
      a = __builtin_fmaf(v.x, v.x, a);
      a = __builtin_fmaf(v.y, v.y, a);
      a = __builtin_fmaf(v.z, v.z, a);
      a = __builtin_fmaf(v.w, v.w, a);
    }
    a = group_sum<16>(a);
    if (gl == 0) out[i] = a;
  }
}

static int idw_check(const char* what, int64_t batches, int64_t rows, int64_t dim) {
  PKM_REQUIRE(batches >= 0 && rows >= 0 && dim > 0, PKM_ERR_INVALID_ARGUMENT, "%s: bad sizes", what);
  PKM_REQUIRE(dim % 4 == 0 && dim < ((int64_t)1 << 30) && batches * rows < ((int64_t)1 << 35), PKM_ERR_UNSUPPORTED,
              "%s: %lld x %lld rows of %lld not supported (rows of whole 16-byte vectors)", what, (long long)batches,
              (long long)rows, (long long)dim);
  return PKM_OK;
}

}  // namespace pkm

using namespace pkm;

extern "C" int pkm_idw_grad_finish(const float* products, const float* x, const float* row_factors, int64_t batches,
                                   int64_t rows, int64_t dim, int row_major, float* out, void* stream) {
  const int rc = idw_check("pkm_idw_grad_finish", batches, rows, dim);
  if (rc != PKM_OK) return rc;
  if (batches * rows == 0) return PKM_OK;
  PKM_REQUIRE(products && x && row_factors && out, PKM_ERR_INVALID_ARGUMENT, "pkm_idw_grad_finish: null pointer");
  PKM_REQUIRE(((uintptr_t)products | (uintptr_t)x | (uintptr_t)out) % 16 == 0, PKM_ERR_INVALID_ARGUMENT,
              "pkm_idw_grad_finish: buffers must be 16-byte aligned");
  const int64_t n = batches * rows * (dim / 4);
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(idw_finish_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0,
                     (hipStream_t)stream, products, x, row_factors, batches, rows, (int)dim, row_major, out);
  return pkm_check_launch("pkm_idw_grad_finish");
}

extern "C" int pkm_row_sumsq(const float* x, int64_t batches, int64_t rows, int64_t dim, int row_major, float* out,
                             void* stream) {
  const int rc = idw_check("pkm_row_sumsq", batches, rows, dim);
  if (rc != PKM_OK) return rc;
  if (batches * rows == 0) return PKM_OK;
  PKM_REQUIRE(x && out, PKM_ERR_INVALID_ARGUMENT, "pkm_row_sumsq: null pointer");
  PKM_REQUIRE((uintptr_t)x % 16 == 0, PKM_ERR_INVALID_ARGUMENT, "pkm_row_sumsq: x must be 16-byte aligned");
  const int64_t blocks = (batches * rows + 15) / 16;
  hipLaunchKernelGGL(row_sumsq_kernel, dim3((unsigned)(blocks < (1 << 20) ? blocks : 1 << 20)), dim3(256), 0,
                     (hipStream_t)stream, x, batches, rows, (int)dim, row_major, out);
  return pkm_check_launch("pkm_row_sumsq");
}

// y = x W^T + b for a few rows, bfloat16, gfx950: the value-side Linears of a
// decode step (pkm/memory.py:222-229) over rows <= 64.
//
// A few rows read W once and multiply it by next to nothing: bound by the
// latency of the W and x loads of a wave, and by the launch. A workgroup of 8
// waves owns 16 outputs; its waves split the inputs, each issuing its loads
// (16-byte fragments of v_mfma_f32_16x16x32_bf16, straight from global memory)
// before its first product; the float32 partial tiles meet in LDS, are summed
// in wave order, get the bias and are rounded once. 8 rows, 1024 x 1024: 3.4 us
// where the BLAS call took 5.3 us on the GPU and 27 us of host time a call; at
// 64 rows 6.8 us against 7.5. With many inputs a wave's chain of products is too
// long and the BLAS is ahead (the caller's rule: memory.py, _rows_kernel_sizes).
#include "pkm_common.h"

namespace pkm {

typedef __bf16 lin_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float lin_f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kLinWaves = 8;
constexpr int kLinMaxRows = 64;

// RT row tiles of 16 (rows past the last read the last row, and are not
// stored); grid: one workgroup per 16 outputs. in a multiple of 32, out of 16.
template <int RT>
__global__ __launch_bounds__(64 * kLinWaves) void linear_rows_kernel(const uint16_t* __restrict__ x,
                                                                     const uint16_t* __restrict__ w,
                                                                     const uint16_t* __restrict__ bias, int rows,
                                                                     int in, int out, uint16_t* __restrict__ y) {
  __shared__ __align__(16) float part[kLinWaves][RT][256];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int o0 = (int)blockIdx.x * 16;
  const int steps = in / 32;  // k-steps, dealt to the waves in consecutive runs
  const int s0 = steps * wv / kLinWaves, s1 = steps * (wv + 1) / kLinWaves;
  const uint16_t* wp = w + (int64_t)(o0 + r) * in + 8 * g;
  const uint16_t* xp[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int row = 16 * t + r < rows ? 16 * t + r : rows - 1;
    xp[t] = x + (int64_t)row * in + 8 * g;
  }
  lin_f32x4_t acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) acc[t] = lin_f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int U = 4;  // k-steps in flight
  for (int s = s0; s < s1; s += U) {
    uint4 b[U], a[U][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 32 * (s + u < s1 ? s + u : s1 - 1);  // a step past the run's end is loaded and not multiplied
      b[u] = ld16(wp + k);
#pragma unroll
      for (int t = 0; t < RT; ++t) a[u][t] = ld16(xp[t] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u < s1) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lin_bf16x8_t, a[u][t]),
                                                           __builtin_bit_cast(lin_bf16x8_t, b[u]), acc[t], 0, 0, 0);
      }
    }
  }
  // acc[t][e]: row 16 t + 4 g + e, output o0 + r
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wv][t][(4 * g + e) * 16 + r] = acc[t][e];
  __syncthreads();
  for (int i = threadIdx.x; i < RT * 256; i += 64 * kLinWaves) {
    const int row = i / 16, c = i % 16;
    if (row >= rows) break;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kLinWaves; ++k) s += part[k][i / 256][i % 256];
    if (bias != nullptr) s += bf16_to_f32(bias[o0 + c]);
    y[(int64_t)row * out + o0 + c] = (uint16_t)f32_to_bf16_bits(s);
  }
}

}  // namespace pkm

using namespace pkm;

extern "C" int pkm_linear_rows(const void* x, const void* weight, const void* bias, int64_t rows, int64_t in_features,
                               int64_t out_features, int dtype, void* y, void* stream) {
  PKM_REQUIRE(dtype == PKM_DTYPE_BF16, PKM_ERR_UNSUPPORTED, "pkm_linear_rows: dtype %d not supported (bfloat16 is)",
              dtype);
  PKM_REQUIRE(rows >= 0 && in_features > 0 && out_features > 0, PKM_ERR_INVALID_ARGUMENT, "pkm_linear_rows: bad sizes");
  PKM_REQUIRE(rows <= kLinMaxRows && in_features % 32 == 0 && out_features % 16 == 0 &&
                  in_features < ((int64_t)1 << 20) && out_features < ((int64_t)1 << 24),
              PKM_ERR_UNSUPPORTED,
              "pkm_linear_rows: rows %lld, in %lld, out %lld not supported (rows <= %d, in a multiple of 32, out of 16)",
              (long long)rows, (long long)in_features, (long long)out_features, kLinMaxRows);
  if (rows == 0) return PKM_OK;
  PKM_REQUIRE(x && weight && y, PKM_ERR_INVALID_ARGUMENT, "pkm_linear_rows: null pointer");
  PKM_REQUIRE(((uintptr_t)x | (uintptr_t)weight) % 16 == 0, PKM_ERR_INVALID_ARGUMENT,
              "pkm_linear_rows: x and weight must be 16-byte aligned");
  const dim3 grid((unsigned)(out_features / 16)), block(64 * kLinWaves);
#define PKM_LINEAR(RT_)                                                                                              \
  hipLaunchKernelGGL(linear_rows_kernel<RT_>, grid, block, 0, (hipStream_t)stream, (const uint16_t*)x,                 \
                     (const uint16_t*)weight, (const uint16_t*)bias, (int)rows, (int)in_features, (int)out_features, \
                     (uint16_t*)y)
  if (rows <= 16)
    PKM_LINEAR(1);
  else if (rows <= 32)
    PKM_LINEAR(2);
  else
    PKM_LINEAR(4);
#undef PKM_LINEAR
  return pkm_check_launch("pkm_linear_rows");
}

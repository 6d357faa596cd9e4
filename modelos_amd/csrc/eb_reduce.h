// Shared pieces of the embedding bag's backward (eb_bwd.hip, eb_bwd_small.hip):
// the in-order reduction of a row's sorted occurrences by a lane group, and
// the host interface of the few-lookups plan.
#pragma once

#include "pkm_common.h"

namespace pkm {

constexpr int kHeavyT = 256;  // chunk length and light/heavy row threshold

// ---------------------------------------------------------------------------
// Segmented reduction over sorted occurrences (generic lane groups).
// ---------------------------------------------------------------------------
template <int VPL>
struct BwdUnroll {
  static constexpr int U = VPL >= 8 ? 2 : (VPL >= 4 ? 4 : 8);
};

// acc += sum over sorted occurrences [i_beg, i_end) (in order) of psw[p] * g[p / L];
// with want_dot, gpsw[p] = <wv, g[p / L]> for each of them.
template <typename TW, typename TG, int LPG, int VPL>
__device__ __forceinline__ void reduce_occurrences(uint32_t i_beg, uint32_t i_end, const uint32_t* __restrict__ svals,
                                                   const void* __restrict__ psw, int pdt,
                                                   const TG* __restrict__ g, int64_t D, uint32_t L32,
                                                   int64_t col0, int glane, const float* wv, bool want_dot,
                                                   void* __restrict__ gpsw, float* acc,
                                                   float* __restrict__ dsorted = nullptr) {
  using GT = GradTraits<TW, TG>;
  constexpr int EPV = VecTraits<TW>::EPV;
  constexpr int NE = VPL * EPV;
  constexpr int NV = GT::NV;
  constexpr int U = BwdUnroll<VPL * NV>::U;
  constexpr int VSTRIDE = LPG * EPV;
  for (uint32_t i0 = i_beg; i0 < i_end; i0 += LPG) {
    const int n = (int)((i_end - i0) < (uint32_t)LPG ? (i_end - i0) : (uint32_t)LPG);
    uint32_t my_p = 0, my_b = 0;
    float my_w = 0.f;
    if (glane < n) {
      my_p = svals[i0 + glane];
      my_b = my_p / L32;
      my_w = psw ? load_scalar(psw, pdt, my_p) : 1.f;
    }
    float my_dot = 0.f;
    for (int jj = 0; jj < n; jj += U) {
      uint4 gvec[U][VPL * NV];
      float w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        w[u] = 0.f;
        if (jj + u < n) {
          const uint32_t b = (uint32_t)bcast_i32<LPG>((int)my_b, jj + u);
          w[u] = bcast_f32<LPG>(my_w, jj + u);
          const TG* grow = g + (int64_t)b * D + col0;
#pragma unroll
          for (int v = 0; v < VPL; ++v)
#pragma unroll
            for (int h = 0; h < NV; ++h) gvec[u][v * NV + h] = ld16(grow + v * VSTRIDE + h * (EPV / NV));
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (jj + u < n) {
          float f[NE];
#pragma unroll
          for (int v = 0; v < VPL; ++v) GT::unpack(&gvec[u][v * NV], f + v * EPV);
#pragma unroll
          for (int e = 0; e < NE; ++e) acc[e] = __builtin_fmaf(f[e], w[u], acc[e]);
          if (want_dot) {
            float d = 0.f;
#pragma unroll
            for (int e = 0; e < NE; ++e) d = __builtin_fmaf(wv[e], f[e], d);
            d = group_sum<LPG>(d);
            if (glane == jj + u) my_dot = d;
          }
        }
      }
    }
    if (want_dot && glane < n) {
      if (dsorted != nullptr)
        dsorted[i0 + glane] = my_dot;  // sorted order, scattered by position later
      else
        store_scalar(gpsw, pdt, my_p, my_dot);
    }
  }
}

template <typename TW, int LPG, int VPL>
__device__ __forceinline__ void load_row_f32(const TW* __restrict__ row, int64_t col0, float* f) {
  constexpr int EPV = VecTraits<TW>::EPV;
#pragma unroll
  for (int v = 0; v < VPL; ++v) VecTraits<TW>::unpack(ld16(row + col0 + v * LPG * EPV), f + v * EPV);
}

// acc += partial sums of a heavy row [beg, end) in chunk order.
template <int LPG, int VPL, int EPV>
__device__ __forceinline__ void add_heavy_partials(uint32_t beg, uint32_t end, const float* __restrict__ partials,
                                                   int64_t D, int64_t col0, float* acc) {
  constexpr int VSTRIDE = LPG * EPV;
  const uint32_t c_first = beg / kHeavyT, c_last = (end - 1) / kHeavyT;
#pragma unroll 4
  for (uint32_t c = c_first; c <= c_last; ++c) {
    const int slot = (c == c_first && beg != c * (uint32_t)kHeavyT) ? 1 : 0;
    const float* prow = partials + (2 * (int64_t)c + slot) * D + col0;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
#pragma unroll
      for (int h = 0; h < EPV; h += 4) {
        float f[4];
        VecTraits<float>::unpack(ld16(prow + v * VSTRIDE + h), f);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[v * EPV + h + e] += f[e];
      }
    }
  }
}

// Zeros over p[0, n), piece t of kFillPer x blockDim.x vectors: piece t lies in
// the (t % 8)-th eighth, so that workgroups dealt round-robin to the XCDs write
// one contiguous eighth per XCD (512 MiB: 6.3 TB/s with 1024 threads; a
// grid-stride loop over the whole range 4.4 to 5.3 TB/s).
constexpr int kFillPer = 4;
__device__ __forceinline__ void fill_piece(uint4* p, size_t n, size_t t) {
  const size_t part = (n + 7) / 8, x = t & 7;
  const size_t end = (x + 1) * part < n ? (x + 1) * part : n;
  size_t i = x * part + (t >> 3) * (size_t)(kFillPer * blockDim.x) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kFillPer; ++k, i += blockDim.x)
    if (i < end) st16(p + i, make_uint4(0u, 0u, 0u, 0u));
}
inline unsigned fill_pieces(size_t n, int threads) {
  const size_t per = (size_t)kFillPer * threads;
  return (unsigned)(((n + 7) / 8 + per - 1) / per * 8);
}
// A share of such a fill, by the workgroups from first_block on of a launch
// whose own are the first `blocks` (first_block: a multiple of 8).
struct FillShare {
  uint4* p = nullptr;
  size_t n = 0;
  uint32_t piece0 = 0, first_block = 0, blocks = 0xFFFFFFFFu;
};
__device__ __forceinline__ bool fill_share(const FillShare& f) {  // true: not one of the launch's own workgroups
  if (blockIdx.x < f.blocks) return false;
  if (blockIdx.x >= f.first_block) fill_piece(f.p, f.n, f.piece0 + (blockIdx.x - f.first_block));
  return true;
}

// ---------------------------------------------------------------------------
// The sparse plan (eb_bwd_small.hip): the reduction of the sorted lookups
// without a walk over the table's rows, whose zeros are written beside the
// sort. Taken by the plain, prepared and accumulating backward for few lookups
// whatever the table (sorted by one workgroup, small_sort), and where the lookups
// are at most a fourth of the rows (sorted by the two-level sort). The table
// gradients are the general plan's, bit for bit where that uses no matrix-core
// products.
// Few lookups, general -> sparse, backward: uniform and Zipf(1.1) lookups, 64 to
// 2^20 rows of 32 bytes to 8 KB, were faster in each of 1488 cases, 1.03 to 31
// times (10 x 1000 into 2^9 x 4096 bf16 916 -> 77 us, 64 x 64 into 2^16 x 64 bf16
// 49 -> 26), also where the lookups are far more than the rows. So are lookups that
// all lie in a few rows (1024 x 10 in 34 rows of 300, which the general plan
// reduces on the matrix cores, 8 KB bf16 171 -> 145 us, 4 KB 130 -> 109), except in
// rows of 512 bytes and less, a lane group each (512 bytes, 10 rows of 1000 123 ->
// 148, 51 rows of 200 110 -> 121).
// ---------------------------------------------------------------------------
constexpr int64_t kSmallLookups = 10240;  // (14 bytes of LDS each in the sort)
inline bool small_plan(int64_t N) { return N > 0 && N <= kSmallLookups; }
// skeys / svals [N] <- rows and positions sorted by (row, position), the
// out-of-range lookups last with row K; *nvalid <- lookups in range. With
// fill: fill_bytes (a multiple of 16) of zeros there, by workgroups beside the sort.
int small_sort(const int64_t* idx, int64_t N, int64_t K, uint32_t* skeys, uint32_t* svals, uint32_t* nvalid,
               void* fill, size_t fill_bytes, hipStream_t st);
int sparse_fill(void* fill, size_t fill_bytes, hipStream_t st);
// The rows with lookups into gW (zeroed before, or, with acc, added to), the
// psw-gradients into gpsw, zeros for the out-of-range lookups: those listed in
// `invalid` (the count, then positions), or with NULL the ones the sorted
// lookups end with (small_sort's).
bool sparse_reduce(const GroupCfg& c, int weight_dtype, int grad_dtype, bool acc, const void* W, int64_t K, int64_t D,
                   const void* psw, int pdt, const void* g, int64_t L, const uint32_t* skeys, const uint32_t* svals,
                   const uint32_t* nvalid, int64_t N, const uint32_t* invalid, float* partials, void* gW, void* gpsw,
                   hipStream_t st);

}  // namespace pkm

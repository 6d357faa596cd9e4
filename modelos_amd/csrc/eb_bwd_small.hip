// Embedding-bag backward where the lookups touch few of the table's rows, gfx950.
//
// The general plan (eb_bwd.hip) walks all K rows, and with few lookups most of
// its 15 to 22 launches take a few microseconds on a handful of workgroups.
// Here the table gradient's zeros (what bounds the call: K x D elements at the
// rate of a fill) are written beside the sort, by workgroups of its launches
// that it leaves idle, and the sorted lookups are reduced without the rows:
//   1. up to kSmallLookups one workgroup sorts (row, position) in LDS; above,
//      the two-level sort;
//   2. a wave per kWin sorted lookups (a lane group per lookup where rows are
//      narrow) reduces the runs that start there, in position order, with
//      their psw-gradients; rows of more than kHeavyT lookups leave chunk
//      partials, as in the general plan;
//   3. (more than kHeavyT lookups only) those rows' partials, in chunk order.
// Forward + backward through autograd: 100 bags x 100 into 2^19 x 512 bf16 250 ->
// 105 us, 64 x 64 into 2^16 x 512 bf16 183 -> 102 (host), 12 x 700 into 2^16 x 2048
// bf16 352 -> 104, 8 x 256 into 2^20 x 1024 bf16 521 -> 353 (2 GiB of zeros at 6.4 TB/s).
#include <atomic>
#include <type_traits>

#include "eb_reduce.h"

namespace pkm {

constexpr int kSsThreads = 1024;
constexpr int kSsWaves = kSsThreads / 64;
constexpr int kSsDigits = 256;

__global__ __launch_bounds__(256) void sparse_fill_kernel(uint4* __restrict__ p, size_t n) {
  fill_piece(p, n, blockIdx.x);
}

// Block 0: stable LSD radix sort of (row, position), 8 bits a pass, in LDS, from
// one buffer into the other. Items are dealt wave-major (wave w: items 64 R w
// .. 64 R (w + 1) - 1, R rounds of 64 lanes), so ranks by wave, round and lane
// keep the item order. The rounds are loops, not straight-line code: one
// workgroup that runs its code once waits for every line of it (16 rounds
// unrolled, items in registers: 70 us at 4096 lookups; as loops 17).
// Blocks 8 on: zeros over fill[0, n16).
__global__ __launch_bounds__(kSsThreads) void small_sort_kernel(const int64_t* __restrict__ idx, int N, uint32_t K,
                                                                int passes, uint32_t* __restrict__ skeys,
                                                                uint32_t* __restrict__ svals,
                                                                uint32_t* __restrict__ nvalid,
                                                                uint4* __restrict__ fill, size_t n16) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (blockIdx.x > 0) {
    if (blockIdx.x >= 8) fill_piece(fill, n16, blockIdx.x - 8);
    return;
  }
  uint32_t(*wcnt)[kSsDigits] = (uint32_t(*)[kSsDigits])smem;  // per wave: digit counts, then the digits' places
  uint32_t* wsum = (uint32_t*)(smem + sizeof(uint32_t) * kSsWaves * kSsDigits);  // [4]
  uint32_t* keys = wsum + 4;
  uint32_t* keys2 = keys + N;
  uint16_t* vals = (uint16_t*)(keys2 + N);
  uint16_t* vals2 = vals + N;
  uint16_t* pre = vals2 + N;  // an item's rank among its wave's items of its digit
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int R = (N + kSsThreads - 1) / kSsThreads;
  const int base = w * 64 * R + lane;  // item i of this thread: base + 64 i
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int p = tid; p < N; p += kSsThreads) {
    const int64_t r = idx[p];
    keys[p] = r >= 0 && r < (int64_t)K ? (uint32_t)r : K;
    vals[p] = (uint16_t)p;
  }
#pragma unroll 1
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = 8 * pass;
    for (int d = tid; d < kSsWaves * kSsDigits; d += kSsThreads) ((uint32_t*)wcnt)[d] = 0;
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < R; ++i) {
      const int p = base + 64 * i;
      const bool valid = p < N;
      const uint32_t d = valid ? (keys[p] >> shift) & (kSsDigits - 1) : 0u;
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        const bool on = (d >> bit) & 1u;
        const uint64_t bb = __ballot(on);
        peers &= on ? bb : ~bb;
      }
      const uint32_t rank = (uint32_t)__popcll(peers & below);
      const uint32_t old = wcnt[w][d];
      if (valid) {
        if (rank == 0) wcnt[w][d] = old + (uint32_t)__popcll(peers);
        pre[p] = (uint16_t)(old + rank);
      }
    }
    __syncthreads();
    // digit starts: thread t < 256 owns digit t
    uint32_t tot = 0, incl = 0;
    if (tid < kSsDigits) {
#pragma unroll 4
      for (int q = 0; q < kSsWaves; ++q) tot += wcnt[q][tid];
      incl = tot;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)incl, o);
        if (lane >= o) incl += y;
      }
      if (lane == 63) wsum[w] = incl;
    }
    __syncthreads();
    if (tid < kSsDigits) {
      uint32_t at = incl - tot;
      for (int q = 0; q < w; ++q) at += wsum[q];
#pragma unroll 4
      for (int q = 0; q < kSsWaves; ++q) {
        const uint32_t c = wcnt[q][tid];
        wcnt[q][tid] = at;
        at += c;
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < R; ++i) {
      const int p = base + 64 * i;
      if (p < N) {
        const uint32_t k = keys[p];
        const uint32_t at = wcnt[w][(k >> shift) & (kSsDigits - 1)] + pre[p];
        keys2[at] = k;
        vals2[at] = vals[p];
      }
    }
    __syncthreads();
    uint32_t* const tk = keys;
    keys = keys2;
    keys2 = tk;
    uint16_t* const tv = vals;
    vals = vals2;
    vals2 = tv;
  }
  for (int p = tid; p < N; p += kSsThreads) {
    const uint32_t key = keys[p];
    skeys[p] = key;
    svals[p] = vals[p];
    if (key < K && (p + 1 == N || keys[p + 1] >= K)) *nvalid = (uint32_t)(p + 1);
    if (p == 0 && key >= K) *nvalid = 0u;
  }
}

// [beg, end) of row r in the nv sorted keys.
__device__ __forceinline__ void run_of(const uint32_t* __restrict__ skeys, uint32_t nv, uint32_t r, uint32_t* beg,
                                       uint32_t* end) {
  uint32_t lo = 0, hi = nv;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (skeys[mid] < r)
      lo = mid + 1;
    else
      hi = mid;
  }
  *beg = lo;
  hi = nv;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (skeys[mid] <= r)
      lo = mid + 1;
    else
      hi = mid;
  }
  *end = lo;
}

// The row's float32 sums into gW; ACC: added, rounded, to the gradient there.
template <typename TW, int LPG, int VPL, bool ACC>
__device__ __forceinline__ void store_grad_row(TW* row, int64_t col0, float* acc) {
  constexpr int EPV = VecTraits<TW>::EPV;
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
    TW* o = row + col0 + v * LPG * EPV;
    if constexpr (ACC) {
      float p[EPV];
      VecTraits<TW>::unpack(ld16(o), p);
#pragma unroll
      for (int e = 0; e < EPV; ++e) acc[v * EPV + e] = p[e] + round_to<TW>(acc[v * EPV + e]);
    }
    st16(o, VecTraits<TW>::pack(acc + v * EPV));
  }
}

// Chunk c of kHeavyT sorted lookups: the partial sums of the rows of more than
// kHeavyT lookups in it, by a lane group; or, of rows of 64 VPL SPLIT vectors, its
// share `part` of the columns: the psw-gradients' parts then meet in `dots`
// [SPLIT][kHeavyT] (LDS), for add_chunk_dots.
template <typename TW, typename TG, int LPG, int VPL, int SPLIT = 1>
__device__ __forceinline__ void sparse_heavy_chunk(uint32_t c, int part, float* dots, const TW* __restrict__ W,
                                                   int64_t D, const void* __restrict__ psw, int pdt,
                                                   const TG* __restrict__ g, uint32_t L32,
                                                   const uint32_t* __restrict__ skeys,
                                                   const uint32_t* __restrict__ svals, uint32_t nv, int glane,
                                                   float* __restrict__ partials, void* __restrict__ gpsw,
                                                   uint32_t* seg) {
  constexpr int EPV = VecTraits<TW>::EPV;
  constexpr int NE = VPL * EPV;
  const int64_t col0 = (int64_t)part * VPL * LPG * EPV + (int64_t)glane * EPV;
  const bool want_dot = gpsw != nullptr;
  const uint32_t i_beg = c * kHeavyT;
  seg[0] = seg[1] = seg[2] = seg[3] = 0;  // the rows' ranges in the chunk
  if (i_beg >= nv) return;
  const uint32_t i_end = i_beg + kHeavyT < nv ? i_beg + kHeavyT : nv;
  const uint32_t cand[2] = {skeys[i_beg], skeys[i_end - 1]};
  const uint32_t before = i_beg > 0 ? skeys[i_beg - 1] : 0xFFFFFFFFu, after = i_end < nv ? skeys[i_end] : 0xFFFFFFFFu;
#pragma unroll 1
  for (int t = 0; t < 2; ++t) {
    const uint32_t r = cand[t];
    if (t == 1 && r == cand[0]) break;
    if (before != r && after != r) continue;  // inside the chunk
    uint32_t s_beg = i_beg, s_end = i_end;
    if (cand[0] != cand[1]) {  // the row's first or last place in the chunk
      const uint32_t key = r + (t == 0 ? 1u : 0u);
      uint32_t lo = i_beg, hi = i_end;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (skeys[mid] < key)
          lo = mid + 1;
        else
          hi = mid;
      }
      // more than kHeavyT lookups: the row is also kHeavyT places before its last one, or past its first
      if (t == 0) {
        s_end = lo;
        if (s_end <= (uint32_t)kHeavyT || skeys[s_end - 1 - kHeavyT] != r) continue;
      } else {
        s_beg = lo;
        if (nv - s_beg <= (uint32_t)kHeavyT || skeys[s_beg + kHeavyT] != r) continue;
      }
    } else if (i_end - i_beg < (uint32_t)kHeavyT && (i_beg == 0 || skeys[i_end - 1 - kHeavyT] != r)) {
      continue;  // (the last, shorter chunk)
    }
    if (t == 0) {
      seg[0] = s_beg;
      seg[1] = s_end;
    } else {
      seg[2] = s_beg;
      seg[3] = s_end;
    }
    float wv[NE], acc[NE];
    if (want_dot) load_row_f32<TW, LPG, VPL>(W + (int64_t)r * D, col0, wv);
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = 0.f;
    reduce_occurrences<TW, TG, LPG, VPL>(s_beg, s_end, svals, psw, pdt, g, D, L32, col0, glane, wv, want_dot, gpsw, acc,
                                         SPLIT > 1 ? dots + part * kHeavyT - (int64_t)i_beg : nullptr);
    float* prow = partials + (2 * (int64_t)c + (s_beg > i_beg ? 1 : 0)) * D + col0;
#pragma unroll
    for (int v = 0; v < VPL; ++v)
#pragma unroll
      for (int h = 0; h < EPV; h += 4) st16(prow + v * LPG * EPV + h, VecTraits<float>::pack(acc + v * EPV + h));
  }
}

// The psw-gradients of chunk c's ranges `seg`, their parts added in order.
template <int SPLIT>
__device__ __forceinline__ void add_chunk_dots(uint32_t c, const uint32_t* seg, const float* dots,
                                               const uint32_t* __restrict__ svals, int pdt, int thread,
                                               void* __restrict__ gpsw) {
  for (int i = thread; i < kHeavyT; i += 64 * SPLIT) {
    const uint32_t p = c * kHeavyT + (uint32_t)i;
    if (!((p >= seg[0] && p < seg[1]) || (p >= seg[2] && p < seg[3]))) continue;
    float d = dots[i];
#pragma unroll
    for (int k = 1; k < SPLIT; ++k) d += dots[k * kHeavyT + i];
    store_scalar(gpsw, pdt, svals[p], d);
  }
}

// The end of row r's run, from position end on, LPG lookups a step; stops past
// kHeavyT lookups from beg.
template <int LPG>
__device__ __forceinline__ uint32_t run_end(const uint32_t* __restrict__ skeys, uint32_t nv, uint32_t r, uint32_t beg,
                                            uint32_t end, int lane, int glane) {
  constexpr uint64_t kAll = LPG == 64 ? ~0ull : ((1ull << LPG) - 1ull);
  while (end - beg <= (uint32_t)kHeavyT) {
    const uint32_t q = end + (uint32_t)glane;
    const uint64_t m = (__ballot(q < nv && skeys[q < nv ? q : beg] == r) >> (lane & ~(LPG - 1))) & kAll;
    if (m != kAll) return end + (uint32_t)__builtin_ctzll(~m);
    end += LPG;
  }
  return end;
}

// Narrow rows. Group j < N: sorted lookup j (the first of its run reduces the
// run; an out-of-range one zeros its psw-gradient). Group N + c: heavy chunk c.
template <typename TW, typename TG, int LPG, int VPL>
__global__ __launch_bounds__(256) void sparse_narrow_kernel(const TW* __restrict__ W, int64_t D,
                                                            const void* __restrict__ psw, int pdt,
                                                            const TG* __restrict__ g, uint32_t L32,
                                                            const uint32_t* __restrict__ skeys,
                                                            const uint32_t* __restrict__ svals,
                                                            const uint32_t* __restrict__ nvalid, uint32_t N,
                                                            uint32_t nchunks, float* __restrict__ partials,
                                                            TW* __restrict__ gW, void* __restrict__ gpsw) {
  constexpr int EPV = VecTraits<TW>::EPV;
  constexpr int NE = VPL * EPV;
  constexpr int GPW = 64 / LPG;
  const int lane = threadIdx.x & 63;
  const int glane = lane & (LPG - 1);
  const uint32_t j = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * GPW + lane / LPG;
  const uint32_t nv = *nvalid;
  if (j >= N) {
    uint32_t seg[4];
    if (j < N + nchunks)
      sparse_heavy_chunk<TW, TG, LPG, VPL>(j - N, 0, nullptr, W, D, psw, pdt, g, L32, skeys, svals, nv, glane, partials,
                                           gpsw, seg);
    return;
  }
  const bool want_dot = gpsw != nullptr;
  if (j >= nv) {
    if (want_dot && glane == 0) store_scalar(gpsw, pdt, svals[j], 0.f);
    return;
  }
  const uint32_t r = skeys[j];
  if (j > 0 && skeys[j - 1] == r) return;
  const uint32_t end = run_end<LPG>(skeys, nv, r, j, j + 1, lane, glane);
  if (end - j > (uint32_t)kHeavyT) return;  // by chunks
  const int64_t col0 = (int64_t)glane * EPV;
  float wv[NE], acc[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) acc[e] = 0.f;
  if (want_dot) load_row_f32<TW, LPG, VPL>(W + (int64_t)r * D, col0, wv);
  reduce_occurrences<TW, TG, LPG, VPL>(j, end, svals, psw, pdt, g, D, L32, col0, glane, wv, want_dot, gpsw, acc);
  store_grad_row<TW, LPG, VPL, false>(gW + (int64_t)r * D, col0, acc);
}

// Rows of 64 VPL vectors. Wave j < nwin: the runs that start at the sorted
// lookups [win j, win (j + 1)), streamed in position order, U lookups' rows
// in flight: the 64 lookups from the window's start are held one per lane (one
// coalesced read each of row, position and weight), a run past them (at most
// kHeavyT lookups) goes on in steps of its own. The last workgroups take the
// heavy chunks: of rows of several vectors a lane up to 4 waves a chunk, each a
// share of the columns, whose loads of all 256 lookups would else hang on one
// wave's 1 to 4 in flight (1024 x 10 lookups in rows of 300, 4096 x 8 KB bf16 234
// -> 145 us, in rows of 1000 225 -> 127, 2 KB 103 -> 89).
// The out-of-range lookups' psw-gradients are zeroed on the way: the sorted
// ones past nvalid (small_sort), or the list `invalid`.
// (A wave per lookup pays five dependent reads for each: backward of 262144
// lookups into 2^20 x 1024 bf16 803 us, 624 so.) Windows of 16 lookups, of 4 up to
// kWinFewLookups, where there are too few of the others to fill the chip: 2^20 x
// 1024 bf16, windows of 4 / 16, 4096 lookups 25.7 / 32.0 us, 10240 50.5 / 55.5,
// 65536 154 / 158 (Zipf(1.1) 214 / 204), 262144 374 / 374 (334 / 309); 2^19 x 2048
// f32, 100000 538 / 568 (451 / 436).
constexpr int kWin = 16;
constexpr int kWinFew = 4;
constexpr int64_t kWinFewLookups = 163840;
template <int VPL>
constexpr int kChunkSplit = VPL < 4 ? VPL : 4;  // waves per heavy chunk

// (Waves per SIMD: what the row's registers leave with its loads in flight. Left
// to itself the compiler trades those for one wave more: 10 x 1000 lookups in rows
// of 200 of 512 x 8 KB f32 101 -> 113 us.)
template <typename TW, int VPL>
constexpr int kRunsWaves = VPL * VecTraits<TW>::EPV >= 32 ? 2 : VPL * VecTraits<TW>::EPV >= 16 ? 3 : 8;

template <typename TW, typename TG, int VPL, bool ACC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, kRunsWaves<TW, VPL>))) void sparse_runs_kernel(const TW* __restrict__ W, int64_t D,
                                                          const void* __restrict__ psw, int pdt,
                                                          const TG* __restrict__ g, uint32_t L32,
                                                          const uint32_t* __restrict__ skeys,
                                                          const uint32_t* __restrict__ svals,
                                                          const uint32_t* __restrict__ nvalid, uint32_t N,
                                                          uint32_t nchunks, int win,
                                                          const uint32_t* __restrict__ invalid,
                                                          float* __restrict__ partials, TW* __restrict__ gW,
                                                          void* __restrict__ gpsw) {
  using GT = GradTraits<TW, TG>;
  constexpr int EPV = VecTraits<TW>::EPV;
  constexpr int NE = VPL * EPV;
  constexpr int NV = GT::NV;
  constexpr int U = VPL * NV >= 8 ? 1 : 8 / (VPL * NV);
  constexpr int SPLIT = kChunkSplit<VPL>;
  constexpr uint32_t CPB = 4 / SPLIT;  // chunks per workgroup
  __shared__ float dots[4][kHeavyT];
  const int lane = threadIdx.x & 63;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t nv = *nvalid;
  const uint32_t nwin = (N + win - 1) / win;
  const uint32_t wblocks = (nwin + 3) / 4;
  if (blockIdx.x >= wblocks) {
    uint32_t seg[4] = {0, 0, 0, 0};
    const uint32_t c = (blockIdx.x - wblocks) * CPB + wave / SPLIT;
    float* const cdots = dots[wave / SPLIT * SPLIT];
    if (c < nchunks)
      sparse_heavy_chunk<TW, TG, 64, VPL / SPLIT, SPLIT>(c, (int)(wave % SPLIT), cdots, W, D, psw, pdt, g, L32, skeys,
                                                         svals, nv, lane, partials, gpsw, seg);
    if constexpr (SPLIT > 1) {
      __syncthreads();
      if (gpsw != nullptr)
        add_chunk_dots<SPLIT>(c, seg, cdots, svals, pdt, (int)(wave % SPLIT) * 64 + lane, gpsw);
    }
    return;
  }
  const uint32_t j = blockIdx.x * 4 + wave;
  if (j >= nwin) return;
  const bool want_dot = gpsw != nullptr;
  if (invalid != nullptr && want_dot) {  // the out-of-range lookups, listed (count first) by the sort
    const uint32_t n = invalid[0];
    for (uint32_t i = j * 64 + (uint32_t)lane; i < n; i += nwin * 64) store_scalar(gpsw, pdt, invalid[1 + i], 0.f);
  }
  const uint32_t s0 = j * win;
  const uint32_t q = s0 + (uint32_t)lane;
  const bool in = q < nv;
  const uint32_t at = in ? q : (nv > 0 ? nv - 1 : 0u);
  const uint32_t key = skeys[at];
  const uint32_t prev = skeys[at > 0 ? at - 1 : 0u];
  const uint32_t val = svals[q < N ? q : N - 1];
  if (invalid == nullptr) {
    if (want_dot && lane < win && q >= nv && q < N) store_scalar(gpsw, pdt, val, 0.f);
  }
  if (s0 >= nv) return;
  const float wgt = psw != nullptr && in ? load_scalar(psw, pdt, val) : 1.f;
  const uint32_t bag = in ? val / L32 : 0u;
  // a lane starts a run (or lies past the lookups)
  const uint64_t starts = __ballot(!in || q == 0 || key != prev);
  const uint64_t mine = starts & __ballot(in) & ((1ull << win) - 1ull);
  if (mine == 0) return;
  const int l0 = __builtin_ctzll(mine);
  const int last = 63 - __builtin_clzll(mine);  // the last run's start
  const uint64_t after = starts & (~0ull << (last + 1));  // (last < win)
  int lend = after != 0 ? __builtin_ctzll(after) : 64;
  const uint32_t r_last = (uint32_t)__builtin_amdgcn_readlane((int)key, last);
  uint32_t tail_end = s0 + 64;  // the last run's end, where it leaves the lanes
  if (after == 0) {
    tail_end = run_end<64>(skeys, nv, r_last, s0 + last, s0 + 64, lane, lane);
    if (tail_end - (s0 + last) > (uint32_t)kHeavyT) lend = last;  // by chunks
  }
  const int64_t col0 = (int64_t)lane * EPV;
  float acc[NE], my_dot = 0.f;
#pragma unroll
  for (int e = 0; e < NE; ++e) acc[e] = 0.f;
  uint32_t row = 0;
  for (int p = l0; p < lend; p += U) {
    uint4 gv[U][VPL * NV], wr[U][VPL];
    uint32_t rr[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int pu = p + u < lend ? p + u : lend - 1;  // (a slot past the end is loaded and not used)
      rr[u] = (uint32_t)__builtin_amdgcn_readlane((int)key, pu);
      const uint32_t bb = (uint32_t)__builtin_amdgcn_readlane((int)bag, pu);
      const TG* grow = g + (int64_t)bb * D + col0;
#pragma unroll
      for (int v = 0; v < VPL; ++v)
#pragma unroll
        for (int h = 0; h < NV; ++h) gv[u][v * NV + h] = ld16(grow + v * 64 * EPV + h * (EPV / NV));
      if (want_dot) {
        const TW* wrow = W + (int64_t)rr[u] * D + col0;
#pragma unroll
        for (int v = 0; v < VPL; ++v) wr[u][v] = ld16(wrow + v * 64 * EPV);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (p + u < lend) {
        if ((starts >> (p + u)) & 1ull) {
          if (p + u > l0) store_grad_row<TW, 64, VPL, ACC>(gW + (int64_t)row * D, col0, acc);
          row = rr[u];
#pragma unroll
          for (int e = 0; e < NE; ++e) acc[e] = 0.f;
        }
        const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wgt), p + u));
        float f[NE];
#pragma unroll
        for (int v = 0; v < VPL; ++v) GT::unpack(&gv[u][v * NV], f + v * EPV);
#pragma unroll
        for (int e = 0; e < NE; ++e) acc[e] = __builtin_fmaf(f[e], w, acc[e]);
        if (want_dot) {
          float wv[NE], d = 0.f;
#pragma unroll
          for (int v = 0; v < VPL; ++v) VecTraits<TW>::unpack(wr[u][v], wv + v * EPV);
#pragma unroll
          for (int e = 0; e < NE; ++e) d = __builtin_fmaf(wv[e], f[e], d);
          d = group_sum<64>(d);
          my_dot = lane == p + u ? d : my_dot;
        }
      }
    }
  }
  if (want_dot && lane >= l0 && lane < lend) store_scalar(gpsw, pdt, val, my_dot);
  if (lend == 64 && tail_end > s0 + 64) {
    float wv[NE];
    if (want_dot) load_row_f32<TW, 64, VPL>(W + (int64_t)row * D, col0, wv);
    reduce_occurrences<TW, TG, 64, VPL>(s0 + 64, tail_end, svals, psw, pdt, g, D, L32, col0, lane, wv, want_dot, gpsw,
                                        acc);
  }
  if (lend > l0) store_grad_row<TW, 64, VPL, ACC>(gW + (int64_t)row * D, col0, acc);
}

// Rows of more than kHeavyT lookups: such a run covers a chunk's first lookup;
// the group of the first such chunk sums the run's partials.
template <typename TW, int LPG, int VPL, bool ACC>
__global__ __launch_bounds__(256) void sparse_heavy_rows_kernel(const uint32_t* __restrict__ skeys,
                                                               const uint32_t* __restrict__ nvalid, uint32_t nchunks,
                                                               int64_t D, const float* __restrict__ partials,
                                                               TW* __restrict__ gW) {
  constexpr int EPV = VecTraits<TW>::EPV;
  constexpr int GPW = 64 / LPG;
  const int lane = threadIdx.x & 63;
  const uint32_t c = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * GPW + lane / LPG;
  const uint32_t nv = *nvalid;
  if (c >= nchunks || c * kHeavyT >= nv) return;
  const uint32_t r = skeys[c * kHeavyT];
  // (such a run reaches half a chunk or more past one side)
  const uint32_t lo = c > 0 ? c * kHeavyT - kHeavyT / 2 : 0u, hi = c * kHeavyT + kHeavyT / 2;
  if (!((c > 0 && skeys[lo] == r) || (hi < nv && skeys[hi] == r))) return;
  uint32_t rb, re;
  run_of(skeys, nv, r, &rb, &re);
  if (re - rb <= (uint32_t)kHeavyT || (c > 0 && rb <= (c - 1) * kHeavyT)) return;
  const int64_t col0 = (int64_t)(lane & (LPG - 1)) * EPV;
  float acc[VPL * EPV];
#pragma unroll
  for (int e = 0; e < VPL * EPV; ++e) acc[e] = 0.f;
  add_heavy_partials<LPG, VPL, EPV>(rb, re, partials, D, col0, acc);
  store_grad_row<TW, LPG, VPL, ACC>(gW + (int64_t)r * D, col0, acc);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static size_t small_sort_lds(int64_t N) {
  return sizeof(uint32_t) * (kSsWaves * kSsDigits + 4) + (size_t)N * 14;
}

int small_sort(const int64_t* idx, int64_t N, int64_t K, uint32_t* skeys, uint32_t* svals, uint32_t* nvalid,
               void* fill, size_t fill_bytes, hipStream_t st) {
  // more than 64 KiB of dynamic LDS: enabled once per device (idempotent, so a race only repeats the call)
  static std::atomic<uint64_t> lds_enabled{0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return pkm_set_error(PKM_ERR_HIP, "pkm_eb_bwd: hipGetDevice failed: %s", hipGetErrorString(e));
  const uint64_t bit = 1ull << (dev & 63);
  if (!(lds_enabled.load(std::memory_order_relaxed) & bit)) {
    e = hipFuncSetAttribute((const void*)small_sort_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)small_sort_lds(kSmallLookups));
    if (e != hipSuccess)
      return pkm_set_error(PKM_ERR_HIP, "pkm_eb_bwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
    lds_enabled.fetch_or(bit, std::memory_order_relaxed);
  }
  int bits = 1;  // of the keys 0 .. K
  while (bits < 32 && ((uint64_t)K >> bits) != 0) ++bits;
  const size_t n16 = fill != nullptr ? fill_bytes / 16 : 0;
  hipLaunchKernelGGL(small_sort_kernel, dim3(n16 > 0 ? 8 + fill_pieces(n16, kSsThreads) : 1), dim3(kSsThreads), small_sort_lds(N), st, idx, (int)N,
                     (uint32_t)K, (bits + 7) / 8, skeys, svals, nvalid, (uint4*)fill, n16);
  return PKM_OK;
}

int sparse_fill(void* fill, size_t fill_bytes, hipStream_t st) {
  const size_t n16 = fill_bytes / 16;
  if (n16 == 0) return PKM_OK;
  hipLaunchKernelGGL(sparse_fill_kernel, dim3(fill_pieces(n16, 256)), dim3(256), 0, st, (uint4*)fill, n16);
  return PKM_OK;
}

template <typename TW, typename TG, int LPG, int VPL, bool ACC>
static void launch_sparse(const void* W, int64_t K, int64_t D, const void* psw, int pdt, const void* g, int64_t L,
                         const uint32_t* skeys, const uint32_t* svals, const uint32_t* nvalid, int64_t N,
                         const uint32_t* invalid, float* partials, void* gW, void* gpsw, hipStream_t st) {
  constexpr int64_t GPB = 4 * (64 / LPG);
  const int64_t nchunks = N > kHeavyT ? (N + kHeavyT - 1) / kHeavyT : 0;
  KernelSpan span("eb_bwd_rows", st);
  if constexpr (LPG == 64) {
    const int win = N > kWinFewLookups ? kWin : kWinFew;
    const int64_t cpb = 4 / kChunkSplit<VPL>;
    const int64_t blocks = (nchunks + cpb - 1) / cpb + ((N + win - 1) / win + 3) / 4;
    hipLaunchKernelGGL((sparse_runs_kernel<TW, TG, VPL, ACC>), dim3((unsigned)blocks), dim3(256), 0, st,
                       (const TW*)W, D, psw, pdt, (const TG*)g, (uint32_t)L, skeys, svals, nvalid, (uint32_t)N,
                       (uint32_t)nchunks, win, invalid, partials, (TW*)gW, gpsw);
  } else {
    static_assert(!ACC, "the accumulating reduction runs on 64-lane rows");
    hipLaunchKernelGGL((sparse_narrow_kernel<TW, TG, LPG, VPL>),
                       dim3((unsigned)((N + nchunks + GPB - 1) / GPB)), dim3(256), 0, st, (const TW*)W, D, psw, pdt, (const TG*)g, (uint32_t)L, skeys, svals, nvalid,
                       (uint32_t)N, (uint32_t)nchunks, partials, (TW*)gW, gpsw);
  }
  if (nchunks > 0)
    hipLaunchKernelGGL((sparse_heavy_rows_kernel<TW, LPG, VPL, ACC>), dim3((unsigned)((nchunks + GPB - 1) / GPB)),
                       dim3(256), 0, st, skeys, nvalid, (uint32_t)nchunks, D, (const float*)partials, (TW*)gW);
}

template <typename TW, typename TG>
static bool dispatch_sparse(const GroupCfg& c, bool acc, const void* W, int64_t K, int64_t D, const void* psw, int pdt,
                           const void* g, int64_t L, const uint32_t* skeys, const uint32_t* svals,
                           const uint32_t* nvalid, int64_t N, const uint32_t* invalid, float* partials, void* gW, void* gpsw,
                  hipStream_t st) {
#define PKM_SPARSE_CASE(LPG_, VPL_)                                                                                   \
  if (c.lpg == LPG_ && c.vpl == VPL_) {                                                                              \
    if constexpr (LPG_ == 64 && std::is_same<TW, TG>::value) {                                                       \
      if (acc) {                                                                                                     \
        launch_sparse<TW, TG, LPG_, VPL_, true>(W, K, D, psw, pdt, g, L, skeys, svals, nvalid, N, invalid, partials, gW, gpsw, \
                                               st);                                                                  \
        return true;                                                                                                 \
      }                                                                                                              \
    }                                                                                                                \
    if (acc) return false;                                                                                           \
    launch_sparse<TW, TG, LPG_, VPL_, false>(W, K, D, psw, pdt, g, L, skeys, svals, nvalid, N, invalid, partials, gW, gpsw,    \
                                            st);                                                                     \
    return true;                                                                                                     \
  }
  PKM_SPARSE_CASE(64, 1)
  PKM_SPARSE_CASE(64, 2)
  PKM_SPARSE_CASE(64, 4)
  PKM_SPARSE_CASE(64, 8)
  PKM_SPARSE_CASE(32, 1)
  PKM_SPARSE_CASE(16, 1)
  PKM_SPARSE_CASE(8, 1)
  PKM_SPARSE_CASE(4, 1)
  PKM_SPARSE_CASE(2, 1)
  PKM_SPARSE_CASE(1, 1)
#undef PKM_SPARSE_CASE
  return false;
}

bool sparse_reduce(const GroupCfg& c, int weight_dtype, int grad_dtype, bool acc, const void* W, int64_t K, int64_t D,
                  const void* psw, int pdt, const void* g, int64_t L, const uint32_t* skeys, const uint32_t* svals,
                  const uint32_t* nvalid, int64_t N, const uint32_t* invalid, float* partials, void* gW, void* gpsw,
                  hipStream_t st) {
#define PKM_SPARSE(TW_, TG_) \
  dispatch_sparse<TW_, TG_>(c, acc, W, K, D, psw, pdt, g, L, skeys, svals, nvalid, N, invalid, partials, gW, gpsw, st)
  if (weight_dtype == PKM_DTYPE_F32) return PKM_SPARSE(float, float);
  const bool wide = grad_dtype == PKM_DTYPE_F32;
  if (weight_dtype == PKM_DTYPE_BF16) return wide ? PKM_SPARSE(bf16_t, float) : PKM_SPARSE(bf16_t, bf16_t);
  return wide ? PKM_SPARSE(f16_t, float) : PKM_SPARSE(f16_t, f16_t);
#undef PKM_SPARSE
}

}  // namespace pkm

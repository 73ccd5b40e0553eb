// Work items of the cross-tile flushes (flush_mfma.hip, sweep_split.hip): target tiles and their k ranges, the
// blocks of WT x WT target tiles of one launch and the order in which workgroups take them.
#pragma once

#include "common.h"

namespace {

struct TileFlush {
  int64_t m, n, mt, nt, S0, S1, S_end;
};

__device__ __forceinline__ bool is_target(const TileFlush& g, int64_t I, int64_t J) {
  return I < g.mt && J < g.nt && I + J >= g.S1 && I + J < g.S_end;
}

// k-tile range of the down (phase 0) or right (phase 1) product of tile (I, J): [lo, hi)
__device__ __forceinline__ void tile_range(const TileFlush& g, int phase, int64_t I, int64_t J, int64_t& lo,
                                           int64_t& hi) {
  const int64_t a = phase == 0 ? J : I, b = phase == 0 ? I : J;
  lo = g.S0 - a > 0 ? g.S0 - a : 0;
  hi = g.S1 - a < b ? g.S1 - a : b;
}

// The launch geometry in 32 bits for the kernel's work-item arithmetic (tile counts and stages stay
// below 2^15): the scalar unit compares 32-bit values itself, while 64-bit signed compares go
// through the vector unit and back -- a per-workgroup walk over the row blocks in 64 bits cost
// microseconds beside the MFMA waves of other workgroups.
struct TileGeo32 {
  int mt, nt, S0, S1, S_end;
};

__device__ __forceinline__ bool is_target(const TileGeo32& g, int I, int J) {
  return I < g.mt && J < g.nt && I + J >= g.S1 && I + J < g.S_end;
}

__device__ __forceinline__ void tile_range(const TileGeo32& g, int phase, int I, int J, int& lo, int& hi) {
  const int a = phase == 0 ? J : I, b = phase == 0 ? I : J;
  lo = g.S0 - a > 0 ? g.S0 - a : 0;
  hi = g.S1 - a < b ? g.S1 - a : b;
}

// Workgroups of a launch are exactly the (row block, column block) pairs that can hold targets:
// row block `by` (tile rows WT by ..) spans the column blocks [first, last] below.  Launching no
// empty workgroups matters: the dispatcher hands workgroups to the XCDs and shader engines in
// turn, and a stride of empty ones leaves whole engines idle while others queue.
template <int WT, typename G, typename Int>
__host__ __device__ inline void row_block_span(const G& g, Int by, Int& first, Int& count) {
  const Int I0 = by * WT;
  Int jt_lo = (Int)g.S1 - (I0 + WT - 1);
  if (jt_lo < 0) jt_lo = 0;
  Int jt_hi = (Int)g.S_end - 1 - I0;  // inclusive
  if (jt_hi > (Int)g.nt - 1) jt_hi = (Int)g.nt - 1;
  // a tile with I, J >= S1 receives nothing (its down range needs J < S1, its right range I < S1)
  if (I0 >= (Int)g.S1 && jt_hi > (Int)g.S1 - 1) jt_hi = (Int)g.S1 - 1;
  first = jt_lo / WT;
  count = (I0 < (Int)g.mt && jt_hi >= jt_lo) ? jt_hi / WT - first + 1 : 0;
}

// Order of the work items.  Row blocks are grouped in bands of SR, and a band's items are numbered column
// block by column block (inside a column by row block), so that a run of 16 consecutive items -- which go
// to one XCD, see the kernel -- is about 4 row blocks x 4 column blocks: every L / C row panel and E / U
// column panel the run streams through its L2 serves four of its workgroups (a run along one row block
// shares its row panel 16 ways and no column panel).
// SR is 4 in flush_mfma.hip and 8 on split operands (twice the reuse of a band's column panels: C5a's flushes 38.9 ->
// 38.1 ms, 8192^2's 5.79 -> 5.76; runs of 32 or 64 items, bands of 16, 38.5-39.4).

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ int wave_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d, 64);
    v += lane >= d ? o : 0;
  }
  return v;
}

// The entry of the sequence of counts f(0), f(1), ..., f(n - 1) that holds position k, with k reduced by the
// counts before it; -1 when k lies past the end.  Each lane evaluates one count per pass of 64 (wave-uniform
// result).
template <typename F>
__device__ __forceinline__ int wave_locate(const F& f, int n, int& k) {
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < n; base += 64) {
    const int cnt = base + lane < n ? f(base + lane) : 0;
    const int s = wave_scan(cnt);
    const int tot = __builtin_amdgcn_readfirstlane(__shfl(s, 63, 64));
    if (k < tot) {
      const unsigned long long hit = __ballot(s > k);  // lane 63 at least
      const int j = __builtin_amdgcn_readfirstlane(__builtin_ctzll(hit));
      k -= __builtin_amdgcn_readfirstlane(__shfl(s - cnt, j, 64));
      return base + j;
    }
    k -= tot;
  }
  return -1;
}

// Row block `by` and column block `bx` of work item `item` (false past the last item).  Wave-parallel: a few
// hundred cycles, where a serial walk over the row blocks cost 10-36 thousand per workgroup at 8192^2.
template <int WT, int SR = 4>
__device__ __forceinline__ bool item_block(const TileGeo32& q, int item, int& by, int& bx) {
  const int nby = (q.mt + WT - 1) / WT, nbands = (nby + SR - 1) / SR;
  auto band_items = [&](int band) {
    int tot = 0;
#pragma unroll
    for (int i = 0; i < SR; ++i) {
      int first = 0, count = 0;
      if (band * SR + i < nby) row_block_span<WT>(q, band * SR + i, first, count);
      tot += count;
    }
    return tot;
  };
  int k = item;
  const int band = wave_locate(band_items, nbands, k);
  if (band < 0) return false;
  int f[SR], c[SR], lo = INT32_MAX, hi = 0;  // the band's spans [f, f + c); columns [lo, hi)
#pragma unroll
  for (int i = 0; i < SR; ++i) {
    f[i] = c[i] = 0;
    if (band * SR + i < nby) row_block_span<WT>(q, band * SR + i, f[i], c[i]);
    if (c[i] > 0) {
      lo = f[i] < lo ? f[i] : lo;
      hi = f[i] + c[i] > hi ? f[i] + c[i] : hi;
    }
  }
  auto column_items = [&](int x) {
    int cnt = 0;
#pragma unroll
    for (int i = 0; i < SR; ++i) cnt += lo + x >= f[i] && lo + x < f[i] + c[i] ? 1 : 0;
    return cnt;
  };
  const int x = wave_locate(column_items, hi - lo, k);
  if (x < 0) return false;
  bx = lo + x;
#pragma unroll
  for (int i = 0; i < SR; ++i)
    if (bx >= f[i] && bx < f[i] + c[i]) {
      if (k == 0) {
        by = band * SR + i;
        return true;
      }
      --k;
    }
  return false;
}

// Workgroups (target blocks of WT x WT tiles) of one launch, per batch entry.
template <int WT>
int64_t count_items(const TileFlush& g) {
  const int64_t rows_hi = g.S_end < g.mt ? g.S_end : g.mt;
  int64_t items = 0;
  for (int64_t by = 0; by * WT < rows_hi; ++by) {
    int64_t first, count;
    row_block_span<WT>(g, by, first, count);
    items += count;
  }
  return items;
}

}  // namespace

// Graph indexing on the device: exclusive scan, per-edge destination index,
// stable CSR transpose (LSD radix sort of col_idx) and the deterministic
// degree-binned row partition.
//
// All of these are integer kernels; every output is a pure function of the
// input (no atomics decide positions), so results are bit-identical across
// runs.  LDS integer atomics are used only to count, never to place.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstring>
#include <type_traits>
#include <vector>

#include "tgx_device.h"
#include "tgx_host.h"

namespace tgx {
namespace {

constexpr int kBlock = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;  // 4096 ints per block

template <typename I>
__device__ __forceinline__ int64_t ld_idx(const I* p, int64_t i) {
  return static_cast<int64_t>(p[i]);
}

// Inclusive scan across one 64-lane wave.
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  const int lane = lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    int t = __shfl_up(v, d, kWave);
    if (lane >= d) v += t;
  }
  return v;
}

// Exclusive scan over the block; returns the thread's exclusive prefix and
// writes the block total to *total.
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds4, int* total) {
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  int inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) lds4[wave] = inc;
  __syncthreads();
  int base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    int t = lds4[w];
    if (w < wave) base += t;
    sum += t;
  }
  __syncthreads();
  *total = sum;
  return base + inc - v;
}

__global__ __launch_bounds__(kBlock) void scan_reduce_kernel(
    const int32_t* __restrict__ in, int64_t n, int32_t* __restrict__ partial) {
  __shared__ int lds4[kBlock / kWave];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t idx = base + static_cast<int64_t>(k) * kBlock + threadIdx.x;
    if (idx < n) s += in[idx];
  }
  int total;
  block_exclusive_scan(s, lds4, &total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// Scan of one tile with a per-block carry-in.
__global__ __launch_bounds__(kBlock) void scan_tile_kernel(
    const int32_t* __restrict__ in, int32_t* __restrict__ out, int64_t n,
    const int32_t* __restrict__ carry, int32_t* __restrict__ total_dev) {
  __shared__ int lds4[kBlock / kWave];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile +
                       static_cast<int64_t>(threadIdx.x) * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t idx = base + k;
    v[k] = idx < n ? in[idx] : 0;
    s += v[k];
  }
  int total;
  int prefix = block_exclusive_scan(s, lds4, &total);
  prefix += carry ? carry[blockIdx.x] : 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t idx = base + k;
    if (idx < n) out[idx] = prefix;
    prefix += v[k];
  }
  if (total_dev && blockIdx.x == gridDim.x - 1 && threadIdx.x == kBlock - 1)
    *total_dev = prefix;
}

}  // namespace

size_t scan_scratch_ints(int64_t n) {
  size_t total = 0;
  while (n > kScanTile) {
    n = ceil_div(n, kScanTile);
    total += static_cast<size_t>(n) + 64;
  }
  return total + 64;
}

int scan_exclusive_i32(const int32_t* in, int32_t* out, int64_t n,
                       int32_t* total_dev, int32_t* scratch, hipStream_t stream) {
  if (n <= 0) {
    if (total_dev) TGX_HIP(hipMemsetAsync(total_dev, 0, sizeof(int32_t), stream));
    return TGX_OK;
  }
  const int64_t blocks = ceil_div(n, kScanTile);
  if (blocks == 1) {
    scan_tile_kernel<<<1, kBlock, 0, stream>>>(in, out, n, nullptr, total_dev);
    TGX_LAUNCHED("scan_tile_kernel");
    return TGX_OK;
  }
  int32_t* partial = scratch;
  int32_t* rest = scratch + align_up(static_cast<size_t>(blocks), 64);
  scan_reduce_kernel<<<blocks, kBlock, 0, stream>>>(in, n, partial);
  TGX_LAUNCHED("scan_reduce_kernel");
  int st = scan_exclusive_i32(partial, partial, blocks, nullptr, rest, stream);
  if (st != TGX_OK) return st;
  scan_tile_kernel<<<blocks, kBlock, 0, stream>>>(in, out, n, partial, total_dev);
  TGX_LAUNCHED("scan_tile_kernel");
  return TGX_OK;
}

namespace {

// ---------------------------------------------------------------------------
// destination index: a workgroup per tile of kIndexTile edges.  Each row that
// starts inside the tile marks its first edge (the last of the rows that
// share a start is the one that owns it), the running maximum of the marks
// along the tile is each edge's row, and the tile leaves in coalesced writes
// whatever the rows' lengths are.  Bound by the writes: 16.8M edges of a
// power-law graph, int64 ids, 126 us with one wave per row (a 64-lane wave
// for rows of 16 edges), 45 us here.  Where more than kIndexRows rows start
// inside a tile (mostly empty ones: few edges in many rows, a gap of unused ids)
// its edges search for their rows instead, so no gap is walked: 4M rows between
// two of 4,000 edges 4833 us walked, 21 us searched; 4M rows of 0.1 edges (20,000
// to a tile) 30 us either way, of 0.22 edges 19 walked and 31 searched.
constexpr int kIndexItems = 8;
constexpr int kIndexTile = kBlock * kIndexItems;
constexpr int kIndexRows = 10 * kIndexTile;

// First r in [0, n_rows] with row_ptr[r] >= edge (n_rows + 1 if none), by one
// wave: 64 probes a step, so a million rows take four dependent loads.
template <typename I>
__device__ __forceinline__ int64_t wave_first_row_at(const I* row_ptr, int64_t n_rows,
                                                     int64_t edge) {
  int64_t lo = 0, hi = n_rows + 1;
  while (lo < hi) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t at = lo + lane_id() * step;
    const int less = __popcll(__ballot(at < hi && ld_idx(row_ptr, at) < edge));
    if (less == 0) break;
    const int64_t stop = lo + less * step;
    lo += (less - 1) * step + 1;
    hi = stop < hi ? stop : hi;
  }
  return lo;
}

template <typename I, typename O>
__global__ __launch_bounds__(kBlock) void destination_index_kernel(
    const I* __restrict__ row_ptr, int64_t n_rows, int64_t n_edges, O* __restrict__ out) {
  __shared__ int mark[kIndexTile];
  __shared__ int wave_max[kBlock / kWave];
  __shared__ int64_t bound[2];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kIndexTile;
  const int64_t end = base + kIndexTile < n_edges ? base + kIndexTile : n_edges;
#pragma unroll
  for (int k = 0; k < kIndexItems; ++k) mark[k * kBlock + threadIdx.x] = 0;
  // Rows that start in (base, end), and before them the row that holds the
  // tile's first edge: the last one starting at or before it.
  if (threadIdx.x < 2 * kWave) {
    const int64_t r = wave_first_row_at(row_ptr, n_rows, threadIdx.x < kWave ? base + 1 : end);
    if (lane_id() == 0) bound[threadIdx.x / kWave] = r;
  }
  __syncthreads();
  const int64_t r_first = bound[0], r_end = bound[1];
  // Rows are counted from the one before r_first, which holds the first edge.
  const int64_t row0 = r_first - 1;
  if (r_end - r_first > kIndexRows) {
    // The last row that starts at or before the edge; a step for all of the
    // thread's edges at once.
    const int64_t n = r_end - row0;
    int64_t at[kIndexItems] = {};
    int64_t half = 1;
    while (half < n) half *= 2;
    for (; half > 0; half /= 2) {
#pragma unroll
      for (int k = 0; k < kIndexItems; ++k) {
        const int64_t to = at[k] + half;
        if (to < n && ld_idx(row_ptr, row0 + to) <= base + k * kBlock + threadIdx.x) at[k] = to;
      }
    }
#pragma unroll
    for (int k = 0; k < kIndexItems; ++k) {
      const int64_t e = base + k * kBlock + threadIdx.x;
      int64_t row = row0 + at[k];
      row = row < n_rows ? row : n_rows - 1;
      if (e < end) out[e] = static_cast<O>(row > 0 ? row : 0);
    }
    return;
  }
  for (int64_t r = r_first + threadIdx.x; r < r_end; r += kBlock) {
    const int64_t at = ld_idx(row_ptr, r) - base;
    if (r < n_rows && at >= 0 && at < kIndexTile)
      atomicMax(&mark[at], static_cast<int>(r - row0));
  }
  __syncthreads();
  // Inclusive running maximum: within the thread's items, over the wave, over
  // the waves.
  int v[kIndexItems];
  int top = 0;
#pragma unroll
  for (int k = 0; k < kIndexItems; ++k) {
    top = max(top, mark[threadIdx.x * kIndexItems + k]);
    v[k] = top;
  }
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  int inc = top;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int t = __shfl_up(inc, d, kWave);
    if (lane >= d) inc = max(inc, t);
  }
  if (lane == kWave - 1) wave_max[wave] = inc;
  int before = __shfl_up(inc, 1, kWave);
  if (lane == 0) before = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w)
    if (w < wave) before = max(before, wave_max[w]);
#pragma unroll
  for (int k = 0; k < kIndexItems; ++k)
    mark[threadIdx.x * kIndexItems + k] = max(v[k], before);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kIndexItems; ++k) {
    const int i = k * kBlock + threadIdx.x;
    const int64_t row = row0 + mark[i];
    if (base + i < end) out[base + i] = static_cast<O>(row > 0 ? row : 0);
  }
}

// *bad = 1 when some index lies outside [0, limit) (the caller clears it).
// One tile per workgroup, all of a thread's loads in flight together: bound by
// the read (16.8M int64 indices: 42 us, 3.2 TB/s from HBM; a minimum and a
// maximum reduction per array took 60 us).
constexpr int kRangeItems = 16;
constexpr int kRangeTile = kBlock * kRangeItems;

template <typename I>
__global__ __launch_bounds__(kBlock) void index_range_kernel(const I* __restrict__ idx, int64_t n,
                                                             int64_t limit,
                                                             int32_t* __restrict__ bad) {
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kRangeTile + threadIdx.x;
  int64_t v[kRangeItems];
#pragma unroll
  for (int k = 0; k < kRangeItems; ++k) {
    const int64_t i = first + k * kBlock;
    v[k] = i < n ? ld_idx(idx, i) : -1;
  }
  bool out_of_range = false;
#pragma unroll
  for (int k = 0; k < kRangeItems; ++k)
    out_of_range |= first + k * kBlock < n && (v[k] < 0 || v[k] >= limit);
  if (out_of_range) *bad = 1;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of 32-bit keys with one or two 32-bit payloads.
//
// A pass over `rb` key bits (at most kSortMaxBits; ids of up to 2^11 rows sort
// in one pass, of up to 2^22 in two) is bound by memory: per key it reads the
// key twice (count, scatter) and each payload once and writes them once.  So
// the passes are few and wide, and the scatter orders each tile of kSortTile
// keys in LDS first: a digit's keys leave as one run of consecutive
// addresses.  Counts lie [tile][digit], so they are written and scanned along
// rows.  Against 8-bit passes that scattered every key to memory by itself
// (16.8M edges, 2^20 rows, int64 ids): a pass 168-201 -> 108-126 us, counts and
// their scan 61 -> 33 us, three passes -> two.
constexpr int kSortBlock = 512;
constexpr int kSortWaves = kSortBlock / kWave;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortBlock * kSortItems;   // 8192 keys per workgroup
constexpr int kSortMaxBits = 11;
constexpr int kSortSegment = 64;                     // tiles per count segment

template <typename K>
__device__ __forceinline__ uint32_t key_at(const K* keys, int64_t i) {
  return static_cast<uint32_t>(keys[i]);
}

template <typename K>
__global__ __launch_bounds__(kSortBlock) void radix_count_kernel(
    const K* __restrict__ keys, int64_t n, int shift, int rb, int32_t* __restrict__ counts) {
  __shared__ int local[1 << kSortMaxBits];
  const int digits = 1 << rb;
  for (int d = threadIdx.x; d < digits; d += kSortBlock) local[d] = 0;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSortTile;
  uint32_t key[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = base + r * kSortBlock + threadIdx.x;
    key[r] = idx < n ? key_at(keys, idx) : 0u;
  }
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = base + r * kSortBlock + threadIdx.x;
    if (idx < n) atomicAdd(&local[(key[r] >> shift) & (digits - 1)], 1);
  }
  __syncthreads();
  int32_t* row = counts + static_cast<int64_t>(blockIdx.x) * digits;
  for (int d = threadIdx.x; d < digits; d += kSortBlock) row[d] = local[d];
}

// Exclusive prefix of each digit's counts over the tiles of one segment, in
// place, and the segment's totals.
__global__ __launch_bounds__(kBlock) void radix_segment_kernel(int32_t* __restrict__ counts,
                                                               int nblocks, int digits,
                                                               int32_t* __restrict__ segments) {
  const int d = blockIdx.x * kBlock + threadIdx.x;
  if (d >= digits) return;
  const int b0 = blockIdx.y * kSortSegment;
  const int b1 = min(b0 + kSortSegment, nblocks);
  int run = 0;
  for (int b = b0; b < b1; b += 16) {
    int v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
      v[k] = b + k < b1 ? counts[static_cast<int64_t>(b + k) * digits + d] : 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (b + k < b1) counts[static_cast<int64_t>(b + k) * digits + d] = run;
      run += v[k];
    }
  }
  segments[static_cast<int64_t>(blockIdx.y) * digits + d] = run;
}

// segments[s][d] -> the keys of digit d in earlier segments; first[d] = the
// keys of smaller digits.  One workgroup; thread t owns digits t and t + 1024.
__global__ __launch_bounds__(1024) void radix_base_kernel(int32_t* __restrict__ segments,
                                                          int nseg, int digits,
                                                          int32_t* __restrict__ first) {
  __shared__ int total[1 << kSortMaxBits];
  __shared__ int wave_sum[16];
  for (int d = threadIdx.x; d < digits; d += 1024) {
    int run = 0;
    for (int s = 0; s < nseg; s += 16) {
      int v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k)
        v[k] = s + k < nseg ? segments[static_cast<int64_t>(s + k) * digits + d] : 0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (s + k < nseg) segments[static_cast<int64_t>(s + k) * digits + d] = run;
        run += v[k];
      }
    }
    total[d] = run;
  }
  __syncthreads();
  // Exclusive scan of the totals: thread t holds digits 2t and 2t + 1.
  const int d0 = 2 * threadIdx.x;
  const int x0 = d0 < digits ? total[d0] : 0;
  const int x1 = d0 + 1 < digits ? total[d0 + 1] : 0;
  const int inc = wave_inclusive_scan(x0 + x1);
  if (lane_id() == kWave - 1) wave_sum[threadIdx.x / kWave] = inc;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w)
    if (w < static_cast<int>(threadIdx.x) / kWave) before += wave_sum[w];
  before += inc - (x0 + x1);
  if (d0 < digits) first[d0] = before;
  if (d0 + 1 < digits) first[d0 + 1] = before + x0;
}

// A payload column of the sort: in == null stands for the key's own index.
template <typename P, typename O>
struct SortColumn {
  const P* in;
  O* out;
};

// Places one tile.  Wave w holds the tile's keys [1024 w, 1024 w + 1024) in
// 16 rounds of 64 consecutive ones, and counts its keys of each digit as it
// goes, so a key's rank among its wave's equal digits follows the input's
// order; with the digits' starts and the earlier waves' counts that is its
// place in the tile.  The tile is put in order in LDS (keys, then each
// payload through the same 32 KB) and written from there.
template <typename K, int RB, typename P0, typename O0, typename P1>
__global__ __launch_bounds__(kSortBlock, 4) void radix_scatter_kernel(
    const K* __restrict__ keys_in, int64_t n, int shift, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ segments, const int32_t* __restrict__ digit_first,
    uint32_t* __restrict__ keys_out, SortColumn<P0, O0> c0, SortColumn<P1, int32_t> c1) {
  constexpr int R = 1 << RB;
  constexpr int PerThread = (R + kSortBlock - 1) / kSortBlock;   // digits a thread scans
  static_assert(kSortWaves * R * 2 <= kSortTile * 4, "the wave counts share the tile's LDS");
  __shared__ uint32_t tile[kSortTile];
  __shared__ int place[R];       // digit's first output position less its first place in the tile
  __shared__ int wave_sum[kSortWaves];
  uint16_t* const cnt = reinterpret_cast<uint16_t*>(tile);   // [kSortWaves][R]
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSortTile;
  const int64_t first = base + wave * (kSortItems * kWave) + lane;
  for (int i = threadIdx.x; i < kSortWaves * R / 2; i += kSortBlock) tile[i] = 0;
  uint32_t key[kSortItems];
  int at[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r)
    key[r] = first + r * kWave < n ? key_at(keys_in, first + r * kWave) : 0u;
  __syncthreads();
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const bool valid = first + r * kWave < n;
    const uint32_t digit = (key[r] >> shift) & (R - 1);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const bool bit = (digit >> b) & 1u;
      const uint64_t bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    // One wave's LDS accesses complete in issue order: every lane reads the
    // count before its group's first lane moves it on.
    const int rank = __popcll(peers & below);
    const int seen = valid ? cnt[wave * R + digit] : 0;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0)
      cnt[wave * R + digit] = static_cast<uint16_t>(seen + __popcll(peers));
    __builtin_amdgcn_wave_barrier();
    at[r] = seen + rank;
  }
  __syncthreads();
  // Digit totals, exclusive over the digits; cnt becomes each wave's first
  // place in the tile.
  int sum[PerThread];
  int mine = 0;
#pragma unroll
  for (int k = 0; k < PerThread; ++k) {
    const int d = threadIdx.x * PerThread + k;
    sum[k] = 0;
    if (d < R)
      for (int w = 0; w < kSortWaves; ++w) sum[k] += cnt[w * R + d];
    mine += sum[k];
  }
  const int inc = wave_inclusive_scan(mine);
  if (lane == kWave - 1) wave_sum[wave] = inc;
  __syncthreads();
  int start = inc - mine;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w)
    if (w < wave) start += wave_sum[w];
  const int32_t* const crow = counts + static_cast<int64_t>(blockIdx.x) * R;
  const int32_t* const srow = segments + static_cast<int64_t>(blockIdx.x / kSortSegment) * R;
#pragma unroll
  for (int k = 0; k < PerThread; ++k) {
    const int d = threadIdx.x * PerThread + k;
    if (d < R) {
      place[d] = crow[d] + srow[d] + digit_first[d] - start;
      int run = start;
      for (int w = 0; w < kSortWaves; ++w) {
        const int c = cnt[w * R + d];
        cnt[w * R + d] = static_cast<uint16_t>(run);
        run += c;
      }
      start = run;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r)
    at[r] += cnt[wave * R + ((key[r] >> shift) & (R - 1))];
  __syncthreads();
  const int m = static_cast<int>(n - base < kSortTile ? n - base : kSortTile);
  int to[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r)
    if (first + r * kWave < n) tile[at[r]] = key[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int i = r * kSortBlock + threadIdx.x;
    if (i < m) {
      const uint32_t k = tile[i];
      to[r] = place[(k >> shift) & (R - 1)] + i;
      keys_out[to[r]] = k;
    }
  }
  auto column = [&](auto c) {
    uint32_t val[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      const int64_t idx = first + r * kWave;
      val[r] = idx < n ? (c.in ? static_cast<uint32_t>(c.in[idx]) : static_cast<uint32_t>(idx))
                       : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
      if (first + r * kWave < n) tile[at[r]] = val[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      const int i = r * kSortBlock + threadIdx.x;
      if (i < m) {
        typedef std::remove_reference_t<decltype(*c.out)> O;
        // (A 64-bit column holds ids below 2^31.)
        c.out[to[r]] = static_cast<O>(static_cast<int32_t>(tile[i]));
      }
    }
  };
  column(c0);
  if (c1.out) column(c1);
}

// out[k] for k in [0, n_keys] = number of sorted keys < k (lower bound), i.e.
// the CSR row pointer of the rows the keys name.
template <typename O>
__global__ __launch_bounds__(kBlock) void run_end_fill_kernel(
    const uint32_t* __restrict__ sorted_keys, int64_t n, int64_t n_keys,
    O* __restrict__ row_ptr) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (k > n_keys) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (static_cast<int64_t>(sorted_keys[mid]) < k) lo = mid + 1; else hi = mid;
  }
  row_ptr[k] = static_cast<O>(lo);
}

// col[i] = src[perm[i]]: the source id of each edge in destination order.
template <typename S>
__global__ __launch_bounds__(kBlock) void gather_src_kernel(
    const int32_t* __restrict__ perm, const S* __restrict__ src, int64_t n,
    S* __restrict__ col) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  col[i] = src[perm[i]];
}

// Varlen block-diagonal relation: sequence k owns positions [cu[k], cu[k+1]).
template <typename I>
__global__ __launch_bounds__(kBlock) void varlen_seq_edges_kernel(
    const I* __restrict__ cu, int64_t n_seq, int causal, int32_t* __restrict__ out) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (k >= n_seq) return;
  const int64_t len = ld_idx(cu, k + 1) - ld_idx(cu, k);
  out[k] = static_cast<int32_t>(causal ? len * (len + 1) / 2 : len * len);
}

// One wave per position: row i of sequence k (start s, length L) relates to
// sources s..i (causal) or s..s+L-1; its edges start at the sequence's first
// edge plus the edges of the earlier rows of the same sequence.
template <typename I>
__global__ __launch_bounds__(kBlock) void varlen_rows_kernel(
    const I* __restrict__ cu, int64_t n_seq, const int32_t* __restrict__ seq_edge0,
    int causal, int64_t total, I* __restrict__ row_ptr, I* __restrict__ col) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) +
                      threadIdx.x / kWave;
  if (row >= total) return;
  // Largest k < n_seq with cu[k] <= row (empty sequences share a start).
  int64_t lo = 0, hi = n_seq - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (ld_idx(cu, mid) <= row) lo = mid; else hi = mid - 1;
  }
  const int64_t s = ld_idx(cu, lo);
  const int64_t len = ld_idx(cu, lo + 1) - s;
  const int64_t p = row - s;
  if (p < 0 || p >= len) return;  // only when cu_seqlens is malformed
  const int64_t start = static_cast<int64_t>(seq_edge0[lo]) +
                        (causal ? p * (p + 1) / 2 : p * len);
  const int64_t deg = causal ? p + 1 : len;
  if (lane_id() == 0) {
    row_ptr[row] = static_cast<I>(start);
    if (row == total - 1) row_ptr[total] = static_cast<I>(start + deg);
  }
  for (int64_t j = lane_id(); j < deg; j += kWave) col[start + j] = static_cast<I>(s + j);
}

__global__ __launch_bounds__(kBlock) void invert_kernel(const int32_t* __restrict__ perm,
                                                        int64_t n,
                                                        int32_t* __restrict__ inv_perm) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) inv_perm[perm[i]] = static_cast<int32_t>(i);
}

// ---------------------------------------------------------------------------
// Degree bins.  Tile of kScanTile rows per block, rows owned in blocked order
// (thread t owns rows t*16 .. t*16+15 of the tile).
template <typename I>
__device__ __forceinline__ int degree_bin(const I* row_ptr, int64_t row,
                                          const int64_t* ub, int n_bins) {
  const int64_t d = ld_idx(row_ptr, row + 1) - ld_idx(row_ptr, row);
  int b = 0;
  while (b < n_bins - 1 && d > ub[b]) ++b;
  return b;
}

struct Bounds {
  int64_t ub[8];
};

template <typename I>
__global__ __launch_bounds__(kBlock) void bin_count_kernel(
    const I* __restrict__ row_ptr, int64_t n_rows, Bounds bounds, int n_bins,
    int nblocks, int32_t* __restrict__ counts) {
  __shared__ int c[8];
  if (threadIdx.x < 8) c[threadIdx.x] = 0;
  __syncthreads();
  int local[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile +
                       static_cast<int64_t>(threadIdx.x) * kScanItems;
  for (int k = 0; k < kScanItems; ++k) {
    int64_t row = base + k;
    if (row < n_rows) local[degree_bin(row_ptr, row, bounds.ub, n_bins)]++;
  }
  for (int b = 0; b < n_bins; ++b)
    if (local[b]) atomicAdd(&c[b], local[b]);
  __syncthreads();
  if (threadIdx.x < n_bins)
    counts[static_cast<int64_t>(threadIdx.x) * nblocks + blockIdx.x] = c[threadIdx.x];
}

template <typename I>
__global__ __launch_bounds__(kBlock) void bin_scatter_kernel(
    const I* __restrict__ row_ptr, int64_t n_rows, Bounds bounds, int n_bins,
    int nblocks, const int32_t* __restrict__ offsets, int32_t* __restrict__ rows_out) {
  __shared__ int lds4[kBlock / kWave];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile +
                       static_cast<int64_t>(threadIdx.x) * kScanItems;
  unsigned char bin[kScanItems];
  for (int k = 0; k < kScanItems; ++k) {
    int64_t row = base + k;
    bin[k] = row < n_rows ? degree_bin(row_ptr, row, bounds.ub, n_bins) : 255;
  }
  for (int b = 0; b < n_bins; ++b) {
    int cnt = 0;
    for (int k = 0; k < kScanItems; ++k) cnt += bin[k] == b;
    int total;
    int pos = block_exclusive_scan(cnt, lds4, &total);
    pos += offsets[static_cast<int64_t>(b) * nblocks + blockIdx.x];
    for (int k = 0; k < kScanItems; ++k)
      if (bin[k] == b) rows_out[pos++] = static_cast<int32_t>(base + k);
  }
}

template <typename I>
__global__ __launch_bounds__(kBlock) void split_count_kernel(
    const I* __restrict__ row_ptr, const int32_t* __restrict__ rows, int64_t n,
    int32_t chunk, int32_t* __restrict__ out) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (k >= n) return;
  const int64_t r = rows[k];
  const int64_t d = ld_idx(row_ptr, r + 1) - ld_idx(row_ptr, r);
  out[k] = static_cast<int32_t>((d + chunk - 1) / chunk);
}

}  // namespace
}  // namespace tgx

using namespace tgx;

extern "C" int tgx_destination_index(const void* row_ptr, int idx_bits, int64_t n_rows,
                                     int64_t n_edges, void* out, int out_bits,
                                     void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(out_bits == 32 || out_bits == 64, "out_bits must be 32 or 64");
  TGX_REQUIRE(n_rows >= 0 && n_edges >= 0, "negative size");
  if (n_rows == 0 || n_edges == 0) return TGX_OK;
  TGX_REQUIRE(row_ptr && out, "null pointer");
  TGX_REQUIRE(out_bits == 64 || n_rows <= INT32_MAX, "row ids overflow int32");
  hipStream_t s = as_stream(stream);
  const auto run = [&](const auto* rp, auto* o) {
    destination_index_kernel<<<ceil_div(n_edges, kIndexTile), kBlock, 0, s>>>(rp, n_rows, n_edges,
                                                                              o);
  };
  const auto with_out = [&](const auto* rp) {
    if (out_bits == 32)
      run(rp, static_cast<int32_t*>(out));
    else
      run(rp, static_cast<int64_t*>(out));
  };
  if (idx_bits == 32)
    with_out(static_cast<const int32_t*>(row_ptr));
  else
    with_out(static_cast<const int64_t*>(row_ptr));
  TGX_LAUNCHED("destination_index_kernel");
  return TGX_OK;
}

extern "C" int tgx_index_range(const void* idx, int idx_bits, int64_t n, int64_t limit,
                               int32_t* bad, void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n >= 0 && n / kRangeTile < (int64_t{1} << 31) - 1, "bad size");
  if (n == 0) return TGX_OK;
  TGX_REQUIRE(idx && bad, "null pointer");
  hipStream_t s = as_stream(stream);
  const unsigned blocks = static_cast<unsigned>(ceil_div(n, int64_t{kRangeTile}));
  if (idx_bits == 32)
    index_range_kernel<<<blocks, kBlock, 0, s>>>(static_cast<const int32_t*>(idx), n, limit, bad);
  else
    index_range_kernel<<<blocks, kBlock, 0, s>>>(static_cast<const int64_t*>(idx), n, limit, bad);
  TGX_LAUNCHED("index_range_kernel");
  return TGX_OK;
}

namespace {

// Scratch of one stable sort of n keys with up to two payloads: two key
// buffers, one of each payload (a payload's passes go to and fro between it and
// the output), the tiles' digit counts and their segments.
struct SortScratch {
  uint32_t* keys[2];
  int32_t* tmp[2];
  int32_t *counts, *segments, *digit_first;
};

SortScratch carve_sort(Carve& c, int64_t n) {
  const int64_t nblocks = ceil_div(n, kSortTile);
  const int64_t nseg = ceil_div(nblocks, kSortSegment);
  SortScratch x;
  for (auto& k : x.keys) k = c.take<uint32_t>(n);
  for (auto& t : x.tmp) t = c.take<int32_t>(n);
  x.counts = c.take<int32_t>(nblocks << kSortMaxBits);
  x.segments = c.take<int32_t>((nseg + 1) << kSortMaxBits);
  x.digit_first = x.segments + (nseg << kSortMaxBits);
  return x;
}

int sort_bits(int64_t key_range) {
  int bits = 0;
  while (bits < 32 && (static_cast<int64_t>(1) << bits) < key_range) ++bits;
  return bits;
}
int sort_passes(int64_t key_range) {
  const int bits = sort_bits(key_range);
  return bits == 0 ? 1 : static_cast<int>(ceil_div(bits, kSortMaxBits));
}

// Stable LSD radix sort of keys in [0, key_range): the payload columns follow
// their keys from col.in (null: the key's index) to col.out; c1.out null
// sorts one column.  Pass p writes a payload to its output if an even number of
// passes follow, else to x.tmp, so col.in may be the one that pass 0 does not
// write.  Returns the buffer that holds the sorted keys.
template <typename K, typename P0, typename O0, typename P1>
uint32_t* stable_sort_by_key(const K* keys, int64_t n, int64_t key_range, SortColumn<P0, O0> c0,
                             SortColumn<P1, int32_t> c1, const SortScratch& x, hipStream_t s,
                             int* status) {
  const int nb = static_cast<int>(ceil_div(n, kSortTile));
  const int nseg = static_cast<int>(ceil_div(nb, kSortSegment));
  int32_t* const counts = x.counts;
  int32_t* const segments = x.segments;
  int32_t* const digit_first = x.digit_first;
  const int bits = sort_bits(key_range);
  const int passes = sort_passes(key_range);
  *status = TGX_OK;
  int shift = 0;
  for (int p = 0; p < passes; ++p) {
    // The bits still to sort, spread evenly; few bits take the 6-bit kernel
    // (a wider digit than the key reads zeros).
    const int left = passes - p;
    int rb = (bits - shift + left - 1) / left;
    if (rb < 6) rb = 6;
    const int digits = 1 << rb;
    const bool first = p == 0, last = p == passes - 1;
    uint32_t* const kout = x.keys[p % 2];
    const uint32_t* const kin = first ? nullptr : x.keys[(p - 1) % 2];
    if (first)
      radix_count_kernel<<<nb, kSortBlock, 0, s>>>(keys, n, shift, rb, counts);
    else
      radix_count_kernel<<<nb, kSortBlock, 0, s>>>(kin, n, shift, rb, counts);
    radix_segment_kernel<<<dim3(ceil_div(digits, kBlock), nseg), kBlock, 0, s>>>(
        counts, nb, digits, segments);
    radix_base_kernel<<<1, 1024, 0, s>>>(segments, nseg, digits, digit_first);
    const auto scatter = [&](const auto* ki, auto col0, auto col1) {
      const auto go = [&](auto rbc) {
        radix_scatter_kernel<std::remove_const_t<std::remove_reference_t<decltype(*ki)>>,
                             decltype(rbc)::value>
            <<<nb, kSortBlock, 0, s>>>(ki, n, shift, counts, segments, digit_first, kout, col0,
                                       col1);
      };
      switch (rb) {
        case 6: go(std::integral_constant<int, 6>{}); break;
        case 7: go(std::integral_constant<int, 7>{}); break;
        case 8: go(std::integral_constant<int, 8>{}); break;
        case 9: go(std::integral_constant<int, 9>{}); break;
        case 10: go(std::integral_constant<int, 10>{}); break;
        default: go(std::integral_constant<int, 11>{}); break;
      }
    };
    // The first pass reads the caller's arrays, the last writes them.
    // (A 64-bit output holds 32-bit values until the last pass.)
    int32_t* const o0 = reinterpret_cast<int32_t*>(c0.out);
    const bool to_out = (passes - 1 - p) % 2 == 0;
    int32_t* const mid0 = to_out ? o0 : x.tmp[0];
    int32_t* const out1 = !c1.out ? nullptr : to_out ? c1.out : x.tmp[1];
    const int32_t* const in0 = to_out ? x.tmp[0] : o0;
    const int32_t* const in1 = to_out ? x.tmp[1] : c1.out;
    if (first && last)
      scatter(keys, c0, c1);
    else if (first)
      scatter(keys, SortColumn<P0, int32_t>{c0.in, mid0}, SortColumn<P1, int32_t>{c1.in, out1});
    else if (last)
      scatter(kin, SortColumn<int32_t, O0>{in0, c0.out}, SortColumn<int32_t, int32_t>{in1, out1});
    else
      scatter(kin, SortColumn<int32_t, int32_t>{in0, mid0},
              SortColumn<int32_t, int32_t>{in1, out1});
    if (hipGetLastError() != hipSuccess) {
      set_error("launch of the radix sort failed");
      *status = TGX_INTERNAL;
      return nullptr;
    }
    shift += rb;
  }
  return x.keys[(passes - 1) % 2];
}

size_t transpose_bytes(int64_t n_edges) {
  Carve c{nullptr, 0};
  carve_sort(c, n_edges);
  return align_up(c.used);
}

}  // namespace

extern "C" int tgx_csr_transpose_workspace(int64_t n_dst, int64_t n_src,
                                           int64_t n_edges, size_t* bytes) {
  TGX_REQUIRE(bytes, "null bytes");
  TGX_REQUIRE(n_dst >= 0 && n_src >= 0 && n_edges >= 0, "negative size");
  *bytes = transpose_bytes(n_edges);
  return TGX_OK;
}

template <typename I>
static int transpose_impl(const I* row_ptr, const I* col, int64_t n_dst, int64_t n_src,
                          int64_t E, int32_t* row_ptr_t, int32_t* col_t,
                          int32_t* perm, int32_t* inv_perm, void* ws, size_t ws_bytes,
                          hipStream_t s) {
  const size_t need = transpose_bytes(E);
  TGX_REQUIRE(ws_bytes >= need, "workspace too small: need %zu bytes", need);
  Carve c{static_cast<char*>(ws), ws_bytes};
  int st = TGX_OK;
  const SortScratch x = carve_sort(c, E);
  // Each edge's destination row rides through the sort beside its index (a
  // gather of it through perm afterwards would fetch a line per edge), from the
  // buffer that pass 0 leaves alone.
  int32_t* const erow = sort_passes(n_src) % 2 ? x.tmp[1] : col_t;
  destination_index_kernel<<<ceil_div(E, kIndexTile), kBlock, 0, s>>>(row_ptr, n_dst, E, erow);
  TGX_LAUNCHED("destination_index_kernel");
  const uint32_t* sorted =
      stable_sort_by_key(col, E, n_src, SortColumn<int32_t, int32_t>{nullptr, perm},
                         SortColumn<int32_t, int32_t>{erow, col_t}, x, s, &st);
  if (st != TGX_OK) return st;
  // row_ptr_t = lower bound of every source id in [0, n_src].
  run_end_fill_kernel<int32_t><<<ceil_div(n_src + 1, kBlock), kBlock, 0, s>>>(
      sorted, E, n_src, row_ptr_t);
  TGX_LAUNCHED("run_end_fill_kernel");
  if (inv_perm) {
    invert_kernel<<<ceil_div(E, kBlock), kBlock, 0, s>>>(perm, E, inv_perm);
    TGX_LAUNCHED("invert_kernel");
  }
  return TGX_OK;
}

extern "C" int tgx_csr_transpose(const void* row_ptr, const void* col, int idx_bits,
                                 int64_t n_dst, int64_t n_src, int64_t n_edges,
                                 int32_t* row_ptr_t, int32_t* col_t, int32_t* perm,
                                 int32_t* inv_perm, void* ws, size_t ws_bytes,
                                 void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n_dst >= 0 && n_src >= 0 && n_edges >= 0, "negative size");
  TGX_REQUIRE(n_edges <= INT32_MAX && n_dst <= INT32_MAX && n_src < INT32_MAX,
              "transpose supports < 2^31 edges and nodes");
  TGX_REQUIRE(row_ptr_t, "null row_ptr_t");
  hipStream_t s = as_stream(stream);
  if (n_edges == 0) {
    TGX_HIP(hipMemsetAsync(row_ptr_t, 0, sizeof(int32_t) * (n_src + 1), s));
    return TGX_OK;
  }
  TGX_REQUIRE(row_ptr && col && col_t && perm && ws, "null pointer");
  if (idx_bits == 32)
    return transpose_impl(static_cast<const int32_t*>(row_ptr),
                          static_cast<const int32_t*>(col), n_dst, n_src, n_edges,
                          row_ptr_t, col_t, perm, inv_perm, ws, ws_bytes, s);
  return transpose_impl(static_cast<const int64_t*>(row_ptr),
                        static_cast<const int64_t*>(col), n_dst, n_src, n_edges,
                        row_ptr_t, col_t, perm, inv_perm, ws, ws_bytes, s);
}

// ---------------------------------------------------------------------------
extern "C" int tgx_plan_degree_bins_workspace(int64_t n_rows, int n_bins, size_t* bytes) {
  TGX_REQUIRE(bytes, "null bytes");
  TGX_REQUIRE(n_rows >= 0 && n_bins >= 1 && n_bins <= 8, "n_bins must be in [1, 8]");
  const int64_t nblocks = ceil_div(n_rows, kScanTile) > 0 ? ceil_div(n_rows, kScanTile) : 1;
  Carve c{nullptr, 0};
  c.take<int32_t>(nblocks * n_bins + 64);
  c.take<int32_t>(scan_scratch_ints(nblocks * n_bins));
  *bytes = align_up(c.used);
  return TGX_OK;
}

extern "C" int tgx_plan_degree_bins(const void* row_ptr, int idx_bits, int64_t n_rows,
                                    const int64_t* upper_bounds, int n_bins,
                                    int32_t* rows_out, int64_t* bin_offsets_host,
                                    void* ws, size_t ws_bytes, void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n_bins >= 1 && n_bins <= 8, "n_bins must be in [1, 8]");
  TGX_REQUIRE(upper_bounds && bin_offsets_host, "null host pointer");
  TGX_REQUIRE(n_rows >= 0 && n_rows <= INT32_MAX, "n_rows must fit int32");
  for (int b = 1; b < n_bins; ++b)
    TGX_REQUIRE(upper_bounds[b] > upper_bounds[b - 1], "upper_bounds must ascend");
  if (n_rows == 0) {
    for (int b = 0; b <= n_bins; ++b) bin_offsets_host[b] = 0;
    return TGX_OK;
  }
  TGX_REQUIRE(row_ptr && rows_out && ws, "null pointer");
  size_t need = 0;
  tgx_plan_degree_bins_workspace(n_rows, n_bins, &need);
  TGX_REQUIRE(ws_bytes >= need, "workspace too small: need %zu bytes", need);
  hipStream_t s = as_stream(stream);
  const int nblocks = static_cast<int>(ceil_div(n_rows, kScanTile));
  Carve c{static_cast<char*>(ws), ws_bytes};
  int32_t* counts = c.take<int32_t>(static_cast<int64_t>(nblocks) * n_bins + 64);
  int32_t* scratch = c.take<int32_t>(scan_scratch_ints(static_cast<int64_t>(nblocks) * n_bins));
  Bounds bd{};
  for (int b = 0; b < 8; ++b) bd.ub[b] = b < n_bins ? upper_bounds[b] : INT64_MAX;
  const int64_t cn = static_cast<int64_t>(nblocks) * n_bins;
  if (idx_bits == 32)
    bin_count_kernel<<<nblocks, kBlock, 0, s>>>(static_cast<const int32_t*>(row_ptr),
                                                n_rows, bd, n_bins, nblocks, counts);
  else
    bin_count_kernel<<<nblocks, kBlock, 0, s>>>(static_cast<const int64_t*>(row_ptr),
                                                n_rows, bd, n_bins, nblocks, counts);
  TGX_LAUNCHED("bin_count_kernel");
  // Per-bin starts are read at counts[b * nblocks] after the scan; the total
  // lands at counts[cn].
  int st = scan_exclusive_i32(counts, counts, cn, counts + cn, scratch, s);
  if (st != TGX_OK) return st;
  if (idx_bits == 32)
    bin_scatter_kernel<<<nblocks, kBlock, 0, s>>>(static_cast<const int32_t*>(row_ptr),
                                                  n_rows, bd, n_bins, nblocks, counts,
                                                  rows_out);
  else
    bin_scatter_kernel<<<nblocks, kBlock, 0, s>>>(static_cast<const int64_t*>(row_ptr),
                                                  n_rows, bd, n_bins, nblocks, counts,
                                                  rows_out);
  TGX_LAUNCHED("bin_scatter_kernel");
  std::vector<int32_t> starts(n_bins + 1);
  for (int b = 0; b < n_bins; ++b)
    TGX_HIP(hipMemcpyAsync(&starts[b], counts + static_cast<int64_t>(b) * nblocks,
                           sizeof(int32_t), hipMemcpyDeviceToHost, s));
  TGX_HIP(hipMemcpyAsync(&starts[n_bins], counts + cn, sizeof(int32_t),
                         hipMemcpyDeviceToHost, s));
  TGX_HIP(hipStreamSynchronize(s));
  for (int b = 0; b <= n_bins; ++b) bin_offsets_host[b] = starts[b];
  if (bin_offsets_host[n_bins] != n_rows) {
    set_error("row partition lost rows: %lld of %lld",
              static_cast<long long>(bin_offsets_host[n_bins]),
              static_cast<long long>(n_rows));
    return TGX_INVALID_ARGUMENT;
  }
  return TGX_OK;
}

extern "C" int tgx_plan_split_chunks(const void* row_ptr, int idx_bits,
                                     const int32_t* split_rows, int64_t n_split,
                                     int32_t chunk_edges, int32_t* chunk_offsets,
                                     int64_t* n_chunks_host, void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(chunk_edges > 0, "chunk_edges must be positive");
  TGX_REQUIRE(n_chunks_host && chunk_offsets, "null pointer");
  TGX_REQUIRE(n_split >= 0 && n_split <= kScanTile * 4096LL, "too many split rows");
  hipStream_t s = as_stream(stream);
  if (n_split == 0) {
    TGX_HIP(hipMemsetAsync(chunk_offsets, 0, sizeof(int32_t), s));
    *n_chunks_host = 0;
    return TGX_OK;
  }
  TGX_REQUIRE(row_ptr && split_rows, "null pointer");
  if (idx_bits == 32)
    split_count_kernel<<<ceil_div(n_split, kBlock), kBlock, 0, s>>>(
        static_cast<const int32_t*>(row_ptr), split_rows, n_split, chunk_edges,
        chunk_offsets);
  else
    split_count_kernel<<<ceil_div(n_split, kBlock), kBlock, 0, s>>>(
        static_cast<const int64_t*>(row_ptr), split_rows, n_split, chunk_edges,
        chunk_offsets);
  TGX_LAUNCHED("split_count_kernel");
  // Up to one scan tile of split rows the device scan needs no scratch and
  // writes the total in place.  Above that (this call has no workspace
  // argument) the per-row counts come to the host, are scanned there and go
  // back; the host buffer lives until the stream has finished both copies.
  if (n_split <= kScanTile) {
    int st = scan_exclusive_i32(chunk_offsets, chunk_offsets, n_split,
                                chunk_offsets + n_split, nullptr, s);
    if (st != TGX_OK) return st;
    int32_t total = 0;
    TGX_HIP(hipMemcpyAsync(&total, chunk_offsets + n_split, sizeof(int32_t),
                           hipMemcpyDeviceToHost, s));
    TGX_HIP(hipStreamSynchronize(s));
    *n_chunks_host = total;
    return TGX_OK;
  }
  std::vector<int32_t> host(n_split + 1);
  TGX_HIP(hipMemcpyAsync(host.data(), chunk_offsets, sizeof(int32_t) * n_split,
                         hipMemcpyDeviceToHost, s));
  TGX_HIP(hipStreamSynchronize(s));
  int64_t run = 0;
  for (int64_t k = 0; k < n_split; ++k) {
    const int32_t v = host[k];
    host[k] = static_cast<int32_t>(run);
    run += v;
  }
  TGX_REQUIRE(run <= INT32_MAX, "chunk count overflows int32");
  host[n_split] = static_cast<int32_t>(run);
  TGX_HIP(hipMemcpyAsync(chunk_offsets, host.data(), sizeof(int32_t) * (n_split + 1),
                         hipMemcpyHostToDevice, s));
  TGX_HIP(hipStreamSynchronize(s));
  *n_chunks_host = run;
  return TGX_OK;
}

// ---------------------------------------------------------------------------
// Graph builders.
namespace {

size_t coo_bytes(int64_t n_edges) {
  Carve c{nullptr, 0};
  carve_sort(c, n_edges);
  return align_up(c.used);
}

template <typename S, typename D>
int coo_impl(const S* src, const D* dst, bool fits32, int64_t n_dst, int64_t E, D* row_ptr,
             S* col, int32_t* perm, void* ws, size_t ws_bytes, hipStream_t s) {
  const size_t need = coo_bytes(E);
  TGX_REQUIRE(ws_bytes >= need, "workspace too small: need %zu bytes", need);
  Carve c{static_cast<char*>(ws), ws_bytes};
  int st = TGX_OK;
  const uint32_t* sorted = nullptr;
  // Sources that fit 32 bits (a 32-bit array, or the caller's word for it) ride
  // through the sort as its payload; others are gathered through the
  // permutation, a line of memory per edge (16.8M edges: 344 us for that gather).
  const bool ride = sizeof(S) == 4 || fits32;
  const SortScratch x = carve_sort(c, E);
  const SortColumn<int32_t, int32_t> order{nullptr, perm};
  if (ride) {
    sorted = stable_sort_by_key(dst, E, n_dst, SortColumn<S, S>{src, col}, order, x, s, &st);
  } else {
    if (!perm) perm = x.tmp[1];   // (one payload: free)
    sorted = stable_sort_by_key(dst, E, n_dst, SortColumn<int32_t, int32_t>{nullptr, perm},
                                SortColumn<int32_t, int32_t>{nullptr, nullptr}, x, s, &st);
  }
  if (st != TGX_OK) return st;
  run_end_fill_kernel<D><<<ceil_div(n_dst + 1, kBlock), kBlock, 0, s>>>(sorted, E, n_dst,
                                                                          row_ptr);
  TGX_LAUNCHED("run_end_fill_kernel");
  if (!ride) {
    gather_src_kernel<S><<<ceil_div(E, kBlock), kBlock, 0, s>>>(perm, src, E, col);
    TGX_LAUNCHED("gather_src_kernel");
  }
  return TGX_OK;
}

template <typename S>
int coo_dispatch_dst(const S* src, const void* dst, int dst_bits, bool fits32, int64_t n_dst,
                     int64_t E, void* row_ptr, void* col, int32_t* perm, void* ws,
                     size_t ws_bytes, hipStream_t s) {
  if (dst_bits == 32)
    return coo_impl(src, static_cast<const int32_t*>(dst), fits32, n_dst, E,
                    static_cast<int32_t*>(row_ptr), static_cast<S*>(col), perm, ws,
                    ws_bytes, s);
  return coo_impl(src, static_cast<const int64_t*>(dst), fits32, n_dst, E,
                  static_cast<int64_t*>(row_ptr), static_cast<S*>(col), perm, ws, ws_bytes,
                  s);
}

int coo_checked(const void* src, int src_bits, const void* dst, int dst_bits, bool fits32,
                int64_t n_dst, int64_t n_edges, void* row_ptr, void* col, int32_t* perm, void* ws,
                size_t ws_bytes, void* stream) {
  TGX_REQUIRE(src_bits == 32 || src_bits == 64, "src_bits must be 32 or 64");
  TGX_REQUIRE(dst_bits == 32 || dst_bits == 64, "dst_bits must be 32 or 64");
  TGX_REQUIRE(n_dst >= 0 && n_edges >= 0, "negative size");
  TGX_REQUIRE(n_edges <= INT32_MAX && n_dst < INT32_MAX,
              "the device builder supports < 2^31 edges and destinations");
  TGX_REQUIRE(row_ptr, "null row_ptr");
  hipStream_t s = as_stream(stream);
  if (n_edges == 0) {
    TGX_HIP(hipMemsetAsync(row_ptr, 0, (dst_bits / 8) * (n_dst + 1), s));
    return TGX_OK;
  }
  TGX_REQUIRE(src && dst && col && ws, "null pointer");
  if (src_bits == 32)
    return coo_dispatch_dst(static_cast<const int32_t*>(src), dst, dst_bits, fits32, n_dst,
                            n_edges, row_ptr, col, perm, ws, ws_bytes, s);
  return coo_dispatch_dst(static_cast<const int64_t*>(src), dst, dst_bits, fits32, n_dst, n_edges,
                          row_ptr, col, perm, ws, ws_bytes, s);
}

size_t varlen_csr_bytes(int64_t n_seq) {
  Carve c{nullptr, 0};
  c.take<int32_t>(n_seq + 1);
  c.take<int32_t>(scan_scratch_ints(n_seq));
  return align_up(c.used);
}

template <typename I>
int varlen_csr_impl(const I* cu, int64_t n_seq, int64_t total, int64_t n_edges, int causal,
                    I* row_ptr, I* col, void* ws, size_t ws_bytes, hipStream_t s) {
  const size_t need = varlen_csr_bytes(n_seq);
  TGX_REQUIRE(ws_bytes >= need, "workspace too small: need %zu bytes", need);
  Carve c{static_cast<char*>(ws), ws_bytes};
  int32_t* edge0 = c.take<int32_t>(n_seq + 1);
  int32_t* scratch = c.take<int32_t>(scan_scratch_ints(n_seq));
  varlen_seq_edges_kernel<I><<<ceil_div(n_seq, kBlock), kBlock, 0, s>>>(cu, n_seq, causal,
                                                                         edge0);
  TGX_LAUNCHED("varlen_seq_edges_kernel");
  int st = scan_exclusive_i32(edge0, edge0, n_seq, edge0 + n_seq, scratch, s);
  if (st != TGX_OK) return st;
  int32_t got = 0;
  TGX_HIP(hipMemcpyAsync(&got, edge0 + n_seq, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  TGX_HIP(hipStreamSynchronize(s));
  TGX_REQUIRE(got == n_edges, "cu_seqlens describe %d edges, caller sized %lld", got,
              static_cast<long long>(n_edges));
  varlen_rows_kernel<I><<<ceil_div(total, kBlock / kWave), kBlock, 0, s>>>(
      cu, n_seq, edge0, causal, total, row_ptr, col);
  TGX_LAUNCHED("varlen_rows_kernel");
  return TGX_OK;
}

}  // namespace

extern "C" int tgx_coo_to_csr_workspace(int64_t n_src, int64_t n_dst, int64_t n_edges,
                                        size_t* bytes) {
  TGX_REQUIRE(bytes, "null bytes");
  TGX_REQUIRE(n_src >= 0 && n_dst >= 0 && n_edges >= 0, "negative size");
  *bytes = coo_bytes(n_edges);
  return TGX_OK;
}

extern "C" int tgx_coo_to_csr(const void* src, int src_bits, const void* dst, int dst_bits,
                              int64_t n_src, int64_t n_dst, int64_t n_edges, void* row_ptr,
                              void* col, int32_t* perm, void* ws, size_t ws_bytes,
                              void* stream) {
  TGX_REQUIRE(n_src >= 0, "negative size");
  return coo_checked(src, src_bits, dst, dst_bits, false, n_dst, n_edges, row_ptr, col, perm, ws,
                     ws_bytes, stream);
}

extern "C" int tgx_coo_to_csr_in_range(const void* src, int src_bits, const void* dst,
                                       int dst_bits, int64_t n_src, int64_t n_dst,
                                       int64_t n_edges, void* row_ptr, void* col, int32_t* perm,
                                       void* ws, size_t ws_bytes, void* stream) {
  TGX_REQUIRE(n_src >= 0, "negative size");
  return coo_checked(src, src_bits, dst, dst_bits, n_src > 0 && n_src <= (int64_t{1} << 31),
                     n_dst, n_edges, row_ptr, col, perm, ws, ws_bytes, stream);
}

extern "C" int tgx_varlen_csr_workspace(int64_t n_seq, size_t* bytes) {
  TGX_REQUIRE(bytes, "null bytes");
  TGX_REQUIRE(n_seq >= 0, "negative size");
  *bytes = varlen_csr_bytes(n_seq);
  return TGX_OK;
}

extern "C" int tgx_varlen_csr(const void* cu_seqlens, int idx_bits, int64_t n_seq,
                              int64_t total, int64_t n_edges, int causal, void* row_ptr,
                              void* col, void* ws, size_t ws_bytes, void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n_seq >= 0 && total >= 0 && n_edges >= 0, "negative size");
  TGX_REQUIRE(n_edges <= INT32_MAX, "the device builder supports < 2^31 edges");
  TGX_REQUIRE(idx_bits == 64 || total <= INT32_MAX, "positions overflow int32");
  TGX_REQUIRE(row_ptr, "null row_ptr");
  hipStream_t s = as_stream(stream);
  if (total == 0 || n_seq == 0) {
    TGX_REQUIRE(total == 0 && n_edges == 0, "no sequences but %lld positions",
                static_cast<long long>(total));
    TGX_HIP(hipMemsetAsync(row_ptr, 0, idx_bits / 8, s));
    return TGX_OK;
  }
  TGX_REQUIRE(cu_seqlens && col && ws, "null pointer");
  if (idx_bits == 32)
    return varlen_csr_impl(static_cast<const int32_t*>(cu_seqlens), n_seq, total, n_edges,
                           causal, static_cast<int32_t*>(row_ptr),
                           static_cast<int32_t*>(col), ws, ws_bytes, s);
  return varlen_csr_impl(static_cast<const int64_t*>(cu_seqlens), n_seq, total, n_edges,
                         causal, static_cast<int64_t*>(row_ptr), static_cast<int64_t*>(col),
                         ws, ws_bytes, s);
}

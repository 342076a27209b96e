// Sum reducer over a destination-row CSR:  out[i, :] = sum_e w[e] * x[col[e], :]
//
// Layout: a gathered row of F features is split into feature tiles of G*VEC
// values; G lanes hold one tile of one edge, 16 bytes per lane (VEC = 4 fp32
// or 8 16-bit values; fewer only where F is smaller), so one wave keeps 64/G
// edges in flight per vector load and U such loads per lane before consuming
// them.  Any F >= VEC takes the 16-byte loads: the last lane of a row moves
// back to the row's last VEC values where F is no multiple of VEC (it repeats
// values of its neighbour, to the bit), and rows need only the alignment of
// their elements.  The edge groups are folded at the end of the row with
// cross-lane adds.
//
// The same kernel is the backward's dx pass: run over the transposed CSR with
// x := dout and the weight fetched through the transpose permutation, it
// computes dx[j] = sum_{e'} w[perm[e']] * dout[col_t[e']] with no atomics.  With
// `self_x` set it also produces dw[perm[e']] = <dout[col_t[e']], x[j]> from the
// row it already holds.
//
// What bounds it: the L2s fetch about 55 G lines a second from beyond
// (Infinity Cache or HBM alike, 64 or 128 bytes of a line alike), 7 TB/s of
// whole lines, and a random row costs the lines it touches.  100,000 rows of
// 16 neighbours, 64 floats: 57 us for 3.2 M lines; 200,000 rows of 12
// neighbours, 100 bf16: 178 us with 8-byte loads, 112 us for 6.1 M lines now.
// (Column tiles of 128 bytes, each XCD's L2 holding one of a 20,000 x 500 table,
// measured slower than whole rows, 60 against 52 us: the edges are then walked 16
// times.)
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "tgx_device.h"
#include "tgx_host.h"
#include "tgx_profile.h"
#include "tgx_tasks.h"

namespace tgx {
namespace {

// VEC consecutive features of one lane: Raw as loaded, widened to fp32 as it
// is consumed.  Weights and the split-row partials are always fp32, and so is
// every sum.  (The vector types claim an element's alignment only; gfx950
// loads and stores 16 bytes at any address.)
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_u __attribute__((ext_vector_type(2), aligned(2)));

template <int DT>
struct Elem;
template <>
struct Elem<TGX_DTYPE_F32> {
  typedef float S;
  static __device__ __forceinline__ float load1(const S* p) { return *p; }
  static __device__ __forceinline__ void store1(S* p, float v) { *p = v; }
};
template <>
struct Elem<TGX_DTYPE_BF16> {
  typedef uint16_t S;
  static __device__ __forceinline__ float load1(const S* p) { return bf16_lo(*p); }
  static __device__ __forceinline__ void store1(S* p, float v) {
    *p = static_cast<uint16_t>(f32_to_bf16_bits(v));
  }
  static __device__ __forceinline__ void widen2(uint32_t w, float* f) {
    f[0] = bf16_lo(w);
    f[1] = bf16_hi(w);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) { return pack_bf16x2(a, b); }
};
template <>
struct Elem<TGX_DTYPE_F16> {
  typedef _Float16 S;
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ float load1(const S* p) { return static_cast<float>(*p); }
  static __device__ __forceinline__ void store1(S* p, float v) { *p = static_cast<_Float16>(v); }
  static __device__ __forceinline__ void widen2(uint32_t w, float* f) {
    const h2 h = __builtin_bit_cast(h2, w);
    f[0] = static_cast<float>(h[0]);
    f[1] = static_cast<float>(h[1]);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, h2{static_cast<_Float16>(a), static_cast<_Float16>(b)});
  }
};

template <int VEC, int DT>
struct Vec {   // 16-bit elements, VEC = 4 or 8
  typedef std::conditional_t<VEC == 8, u32x4_u, u32x2_u> Raw;
  typedef typename Elem<DT>::S S;
  static __device__ __forceinline__ Raw load(const S* p) {
    return *reinterpret_cast<const Raw*>(p);
  }
  static __device__ __forceinline__ void widen(Raw r, float (&f)[VEC]) {
#pragma unroll
    for (int k = 0; k < VEC / 2; ++k) Elem<DT>::widen2(r[k], f + 2 * k);
  }
  static __device__ __forceinline__ void store(S* p, const float (&f)[VEC]) {
    Raw r;
#pragma unroll
    for (int k = 0; k < VEC / 2; ++k) r[k] = Elem<DT>::pack2(f[2 * k], f[2 * k + 1]);
    *reinterpret_cast<Raw*>(p) = r;
  }
};
template <>
struct Vec<4, TGX_DTYPE_F32> {
  typedef f32x4_u Raw;
  typedef float S;
  static __device__ __forceinline__ Raw load(const S* p) {
    return *reinterpret_cast<const Raw*>(p);
  }
  static __device__ __forceinline__ void widen(Raw r, float (&f)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = r[k];
  }
  static __device__ __forceinline__ void store(S* p, const float (&f)[4]) {
    *reinterpret_cast<Raw*>(p) = Raw{f[0], f[1], f[2], f[3]};
  }
};
template <int DT>
struct Vec<1, DT> {
  typedef typename Elem<DT>::S S;
  typedef S Raw;
  static __device__ __forceinline__ Raw load(const S* p) { return *p; }
  static __device__ __forceinline__ void widen(Raw r, float (&f)[1]) {
    f[0] = Elem<DT>::load1(&r);
  }
  static __device__ __forceinline__ void store(S* p, const float (&f)[1]) {
    Elem<DT>::store1(p, f[0]);
  }
};
// A lane's values of a split row's fp32 partial.
template <int VEC>
__device__ __forceinline__ void store_partial(float* p, const float (&f)[VEC]) {
  if constexpr (VEC == 1) {
    p[0] = f[0];
  } else {
#pragma unroll
    for (int k = 0; k < VEC; k += 4)
      *reinterpret_cast<f32x4_u*>(p + k) = f32x4_u{f[k], f[k + 1], f[k + 2], f[k + 3]};
  }
}

template <typename I, int DT>
struct SumArgs {
  typedef typename Elem<DT>::S S;
  const I* row_ptr;
  const I* col;
  PlanView plan;
  const S* x;              // gathered table [*, F]
  const float* w;          // per-edge weight or null (=1)
  const int32_t* wperm;    // weight index = wperm[e] when non-null
  S* out;                  // [rows, F]
  float* partial;          // [n_chunks, F]
  const S* self_x;         // dw: row's own features [rows, F] (null = no dw)
  float* dw;               // dw output, written at dwperm ? dwperm[e] : e
  const int32_t* dwperm;
  int64_t F;
  int64_t dw_tile;         // floats between the feature tiles' dw (dw sums of one tile each)
};

// A lane's features of the tile: the offset of its VEC values in a row, and
// how many of them its neighbour holds too (a moved last lane).
struct LaneCols {
  int64_t at;
  int repeated;
  bool active;
};
template <int VEC>
__device__ __forceinline__ LaneCols lane_cols(int64_t first, int64_t F) {
  LaneCols l{first, 0, first < F};
  if constexpr (VEC > 1) {
    l.at = first < F - VEC ? first : F - VEC;
    l.repeated = static_cast<int>(first - l.at);
  }
  return l;
}

// The row's own values for dw; repeated ones count once.
template <int VEC, int DT>
__device__ __forceinline__ void load_self(const typename Elem<DT>::S* row, const LaneCols& l,
                                          float (&self)[VEC]) {
  Vec<VEC, DT>::widen(Vec<VEC, DT>::load(row + l.at), self);
#pragma unroll
  for (int k = 0; k < VEC; ++k)
    if (k < l.repeated) self[k] = 0.f;
}

template <int VEC>
__device__ __forceinline__ float dot(const float (&a)[VEC], const float (&b)[VEC]) {
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < VEC; ++k) s += a[k] * b[k];
  return s;
}

// A second look at the dw of edges e, e + step, ... < e1 of a row, where some
// came out NaN: an infinite repeated value times the 0 of load_self is NaN where
// the sum may be Inf.  Those are formed again from the two rows' columns
// [first, end), each once.  (The gather loops only note that there is one, and
// launches without dw have kernels of their own: fp16 F = 11, 2.7M edges fwd +
// bwd 232 us before this, 230 so; with a select per gathered value, or all of it
// in one kernel, 244.)
template <typename I, int DT>
__device__ __forceinline__ void redo_nan_dw(const SumArgs<I, DT>& a, int64_t row, int64_t e,
                                            int64_t e1, int step, int64_t dw_off, int64_t first,
                                            int64_t end) {
  const typename Elem<DT>::S* const self = a.self_x + row * a.F;
#pragma unroll 1
  for (; e < e1; e += step) {
    float* const to = a.dw + dw_off + (a.dwperm ? static_cast<int64_t>(a.dwperm[e]) : e);
    if (*to == *to) continue;
    const typename Elem<DT>::S* const x = a.x + (a.col ? static_cast<int64_t>(a.col[e]) : e) * a.F;
    float s = 0.f;
#pragma unroll 1
    for (int64_t k = first; k < end; ++k) s += Elem<DT>::load1(x + k) * Elem<DT>::load1(self + k);
    *to = s;
  }
}

// One whole-wave task (a row, a split-row chunk or a group of empty rows).
template <typename I, int DT, int VEC, int G, int U, bool DW>
__device__ __forceinline__ void sum_task(const SumArgs<I, DT>& a, const Task& t, int tile,
                                         float* dw_stage) {
  typedef Vec<VEC, DT> V;
  constexpr int EPW = kWave / G;  // edges per wave-wide load
  if (t.kind == kTaskNone) return;
  const int lane = lane_id();
  const int g = lane / G;
  const int c = lane % G;
  const int64_t F = a.F;
  const LaneCols lc = lane_cols<VEC>(static_cast<int64_t>(tile) * (G * VEC) + c * VEC, F);

  if (t.kind == kTaskEmpty) {
    for (int k = 0; k < t.n_empty; ++k) {
      const int row = uniform(a.plan.rows[t.empty0 + k]);
      const float zero[VEC] = {};
      if (g == 0 && lc.active && a.out)
        V::store(a.out + static_cast<int64_t>(row) * F + lc.at, zero);
    }
    return;
  }

  float self[VEC] = {};
  if (DW && lc.active)
    load_self<VEC, DT>(a.self_x + static_cast<int64_t>(t.row) * F, lc, self);

  float acc[VEC] = {};
  bool nan = false;   // this lane wrote a dw that is NaN
  for (int64_t base = t.e0; base < t.e1; base += kWave) {
    const int n = static_cast<int>(t.e1 - base < kWave ? t.e1 - base : kWave);
    int my_col = 0;
    float my_w = 0.f;
    int my_wp = 0;   // wperm[e] (int32: a permuted relation has < 2^31 edges)
    if (lane < n) {
      // No column array: the columns are the edge ids (a per-edge field
      // summed per row, read contiguously).
      const int64_t e = base + lane;
      my_col = a.col ? static_cast<int>(a.col[e]) : static_cast<int>(e);
      if (a.wperm) my_wp = a.wperm[e];
      my_w = a.w ? a.w[a.wperm ? static_cast<int64_t>(my_wp) : e] : 1.f;
    }
    for (int k = 0; k < n; k += EPW * U) {
      typename V::Raw v[U];
      float wt[U];
      int slot[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        slot[u] = k + u * EPW + g;
        const int src = slot[u] < n ? slot[u] : 0;
        const int j = __shfl(my_col, src, 64);
        wt[u] = __shfl(my_w, src, 64);
        v[u] = typename V::Raw{};
        if (slot[u] < n && lc.active) v[u] = V::load(a.x + static_cast<int64_t>(j) * F + lc.at);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float f[VEC];
        V::widen(v[u], f);
        if (slot[u] < n) {
#pragma unroll
          for (int q = 0; q < VEC; ++q) acc[q] += wt[u] * f[q];
        }
        if constexpr (DW) {
          const float d = group_sum<G>(dot(f, self));
          if (c == 0 && slot[u] < n) dw_stage[slot[u]] = d;
        }
      }
    }
    if constexpr (DW) {
      // A window's dw values wait in LDS and leave with one store per lane
      // after the window, not one store per edge group inside the gather loop
      // (whose following gathers would share its in-order completion count).
      // One wave's LDS accesses complete in issue order: lane e reads the
      // value another lane wrote for edge base + e.
      __builtin_amdgcn_wave_barrier();
      if (lane < n) {
        const int64_t at = a.dwperm ? static_cast<int64_t>(a.wperm ? my_wp : a.dwperm[base + lane])
                                    : base + lane;
        const float d = dw_stage[lane];
        a.dw[tile * a.dw_tile + at] = d;
        nan |= d != d;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  if constexpr (DW && VEC > 1) {
    if (F % VEC != 0 && __any(nan)) {
      const int64_t first = static_cast<int64_t>(tile) * (G * VEC);
      redo_nan_dw(a, t.row, t.e0 + lane, t.e1, kWave, tile * a.dw_tile, first,
                  first + G * VEC < F ? first + G * VEC : F);
    }
  }
  // Fold the EPW edge groups (lanes with equal c).
#pragma unroll
  for (int m = G; m < kWave; m <<= 1)
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[q] += __shfl_xor(acc[q], m, 64);
  // A null out: only the per-edge dot products (dw) are wanted.
  if (g != 0 || !lc.active || !a.out) return;
  if (t.kind == kTaskChunk)
    store_partial<VEC>(a.partial + static_cast<int64_t>(t.slot) * F + lc.at, acc);
  else
    V::store(a.out + static_cast<int64_t>(t.row) * F + lc.at, acc);
}

template <typename I, int DT, int VEC, int G, int U, bool DW>
__global__ __launch_bounds__(kTaskBlock) void sum_rows_kernel(SumArgs<I, DT> a) {
  __shared__ float dw_stage[kWavesPerBlock][kWave];
  sum_task<I, DT, VEC, G, U, DW>(a, decode_task(a.plan, a.row_ptr, global_wave()), blockIdx.y,
                             dw_stage[threadIdx.x / kWave]);
}

// Narrow tiles (G <= 8 lanes per edge): the wave splits into 64 / SLOT lane
// slots of SLOT lanes, each taking P rows of the wave bin, so a wave's fixed
// cost (task decode, the dependent row_ptr -> col -> gather chain) covers
// (64 / SLOT) P rows, and the loads of a slot's P rows are in flight
// together.  A slot keeps U SLOT / G edges per row in flight.  The task list is
//   [split-row chunks | row groups | empty-row groups];
// chunks and empty groups run as whole-wave tasks, and after the group's other
// rows so does each row of over kSlotRow edges.  Slot s of group w takes the
// wave-bin rows S P w + S q + s, q < P, S = 64 / SLOT.
template <int SLOT>
constexpr int kSlotRow = 4 * SLOT;

template <typename I, int DT, int VEC, int G, int UC, int SLOT, int P, int U, bool DW>
__global__ __launch_bounds__(kTaskBlock) void sum_pairs_kernel(SumArgs<I, DT> a) {
  typedef Vec<VEC, DT> V;
  constexpr int NS = kWave / SLOT;   // slots per wave
  constexpr int EPH = SLOT / G;      // edges per slot load
  __shared__ float dw_stage[kWavesPerBlock][P * kWave];
  const PlanView& p = a.plan;
  const int wv = threadIdx.x / kWave;
  float* const stage = dw_stage[wv];
  const int64_t w = global_wave();
  const int64_t n_groups = (p.n_wave + NS * P - 1) / (NS * P);
  const int64_t pw = w - p.n_chunks;
  if (pw < 0 || pw >= n_groups) {
    sum_task<I, DT, VEC, G, UC, DW>(
        a, decode_task(p, a.row_ptr, pw < 0 ? w : p.n_chunks + p.n_wave + (pw - n_groups)), 0,
        stage);
    return;
  }
  const int lane = lane_id();
  const int slot_id = lane / SLOT, hl = lane % SLOT;
  const int g = hl / G, c = hl % G;
  const int64_t F = a.F;
  const LaneCols lc = lane_cols<VEC>(c * VEC, F);   // (one tile)
  int row[P], len[P];
  int64_t e0[P];
  bool has[P];      // rows the slots sum here
  uint64_t late[P]; // lanes of the slots whose row runs whole-wave afterwards
  int len_max = 0;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int64_t k = NS * P * pw + NS * q + slot_id;   // position in the wave bin
    has[q] = k < p.n_wave;
    row[q] = has[q] ? p.rows[p.n_empty + k] : 0;
    e0[q] = has[q] ? static_cast<int64_t>(a.row_ptr[row[q]]) : 0;
    len[q] = has[q] ? static_cast<int>(static_cast<int64_t>(a.row_ptr[row[q] + 1]) - e0[q]) : 0;
    late[q] = __ballot(hl == 0 && len[q] > kSlotRow<SLOT>);
    if (len[q] > kSlotRow<SLOT>) {
      has[q] = false;
      len[q] = 0;
    }
    len_max = max(len_max, len[q]);
  }
  // Every slot loops to the longest row (wave-uniform bounds keep every
  // shuffle's source lanes active); each row masks its own tail.
#pragma unroll
  for (int m = SLOT; m < kWave; m <<= 1) len_max = max(len_max, __shfl_xor(len_max, m, 64));
  len_max = uniform(len_max);
  float self[P][VEC] = {}, acc[P][VEC] = {};
  bool nan = false;
#pragma unroll
  for (int q = 0; q < P; ++q)
    if (DW && lc.active && has[q])
      load_self<VEC, DT>(a.self_x + static_cast<int64_t>(row[q]) * F, lc, self[q]);
  for (int base = 0; base < len_max; base += SLOT) {
    int n[P], my_col[P], my_wp[P];
    float my_w[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
      n[q] = min(max(len[q] - base, 0), SLOT);   // this row's edges
      my_col[q] = 0;
      my_wp[q] = 0;
      my_w[q] = 0.f;
      if (hl < n[q]) {
        const int64_t e = e0[q] + base + hl;
        my_col[q] = a.col ? static_cast<int>(a.col[e]) : static_cast<int>(e);
        if (a.wperm) my_wp[q] = a.wperm[e];
        my_w[q] = a.w ? a.w[a.wperm ? static_cast<int64_t>(my_wp[q]) : e] : 1.f;
      }
    }
    const int n_max = min(len_max - base, SLOT);   // wave-uniform
    for (int kk = 0; kk < n_max; kk += EPH * U) {
      typename V::Raw v[P][U];
      float wt[P][U];
      int slot[U];
#pragma unroll
      for (int u = 0; u < U; ++u) slot[u] = kk + u * EPH + g;
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int src = SLOT * slot_id + (slot[u] < n[q] ? slot[u] : 0);
          const int j = __shfl(my_col[q], src, 64);
          wt[q][u] = __shfl(my_w[q], src, 64);
          v[q][u] = typename V::Raw{};
          if (slot[u] < n[q] && lc.active)
            v[q][u] = V::load(a.x + static_cast<int64_t>(j) * F + lc.at);
        }
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float f[VEC];
          V::widen(v[q][u], f);
          if (slot[u] < n[q]) {
#pragma unroll
            for (int r = 0; r < VEC; ++r) acc[q][r] += wt[q][u] * f[r];
          }
          if constexpr (DW) {
            const float d = group_sum<G>(dot(f, self[q]));
            if (c == 0 && slot[u] < n[q]) stage[q * kWave + SLOT * slot_id + slot[u]] = d;
          }
        }
    }
    if constexpr (DW) {
      // (As in sum_task: dw leaves after the window, one store per lane.)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < P; ++q)
        if (hl < n[q]) {
          const int64_t e = e0[q] + base + hl;
          const int64_t at = a.dwperm ? static_cast<int64_t>(a.wperm ? my_wp[q] : a.dwperm[e]) : e;
          const float d = stage[q * kWave + lane];
          a.dw[at] = d;
          nan |= d != d;
        }
      __builtin_amdgcn_wave_barrier();
    }
  }
  if constexpr (DW && VEC > 1) {
    if (F % VEC != 0 && __any(nan)) {
#pragma unroll
      for (int q = 0; q < P; ++q)
        redo_nan_dw(a, row[q], e0[q] + hl, e0[q] + len[q], SLOT, 0, 0, F);
    }
  }
  // Fold each row's edge groups (lanes with equal c; masks below SLOT stay
  // inside the slot).
#pragma unroll
  for (int q = 0; q < P; ++q) {
#pragma unroll
    for (int m = G; m < SLOT; m <<= 1)
#pragma unroll
      for (int r = 0; r < VEC; ++r) acc[q][r] += __shfl_xor(acc[q][r], m, 64);
    if (g == 0 && lc.active && has[q] && a.out)
      V::store(a.out + static_cast<int64_t>(row[q]) * F + lc.at, acc[q]);
  }
#pragma unroll
  for (int q = 0; q < P; ++q)
    for (uint64_t m = late[q]; m; m &= m - 1) {
      const int64_t k = NS * P * pw + NS * q + (__ffsll(static_cast<long long>(m)) - 1) / SLOT;
      sum_task<I, DT, VEC, G, UC, DW>(a, decode_task(p, a.row_ptr, p.n_chunks + k), 0, stage);
    }
}

// Combine split-row chunk partials in chunk order (deterministic).
template <int DT>
__global__ __launch_bounds__(kTaskBlock) void sum_merge_kernel(
    PlanView plan, const float* __restrict__ partial, typename Elem<DT>::S* __restrict__ out,
    int64_t F) {
  const int64_t k = global_wave();
  if (k >= plan.n_split) return;
  const int row = uniform(plan.rows[plan.n_empty + plan.n_wave + k]);
  const int c0 = plan.chunk_off[k], c1 = plan.chunk_off[k + 1];
  for (int64_t f = lane_id(); f < F; f += kWave) {
    float s = 0.f;
    for (int c = c0; c < c1; ++c) s += partial[static_cast<int64_t>(c) * F + f];
    Elem<DT>::store1(out + static_cast<int64_t>(row) * F + f, s);
  }
}

template <typename I, int DT, int VEC, int G>
void launch_sum(const SumArgs<I, DT>& a, int tiles, hipStream_t s) {
  constexpr int U = (kWave / G) >= 16 ? 1 : (16 / (kWave / G) < 8 ? 16 / (kWave / G) : 8);
  const PlanView& p = a.plan;
  // Rows of up to 8 lanes share a wave: they are short in time, so a row's fixed
  // cost weighs more.  Not rows of 16 lanes: four to a wave gain nothing on even
  // degrees (bf16 F = 100, 12-edge rows 112 us, 111 one a wave) and a wave of
  // several long rows ends late (R-MAT, 262,144 rows of 16 edges 188 against 132,
  // 16,384 rows of 32 edges 68 against 33).
  if constexpr (G <= 8) {
    // One lane per edge: 16-lane slots of 2 rows each, 8 rows per wave (the
    // reference's F = 1 case, 131072 rows of 16 edges: 0.0254 ms with 32-lane
    // slots of 2 rows, 0.0182 ms with these).  2 to 8 lanes: 32-lane slots of
    // one row (two rows per wave measured 5% faster than four on 8-wide rows;
    // 8 lanes, bf16 F = 64, 16-edge rows 36 us against 43 one a wave, though
    // R-MAT 111 against 102).
    constexpr int SLOT = G == 1 ? 16 : 32;
    constexpr int P = G == 1 ? 2 : 1;
    constexpr int NS = kWave / SLOT;
    const int64_t waves = p.n_chunks + (p.n_wave + NS * P - 1) / (NS * P) +
                          (p.n_empty + kEmptyPerWave - 1) / kEmptyPerWave;
    const auto k = a.self_x ? sum_pairs_kernel<I, DT, VEC, G, U, SLOT, P, G, true>
                            : sum_pairs_kernel<I, DT, VEC, G, U, SLOT, P, G, false>;
    k<<<static_cast<unsigned>(ceil_div(waves, kWavesPerBlock)), kTaskBlock, 0, s>>>(a);
  } else {
    const dim3 grid(static_cast<unsigned>(ceil_div(plan_waves(p), kWavesPerBlock)),
                    static_cast<unsigned>(tiles));
    const auto k = a.self_x ? sum_rows_kernel<I, DT, VEC, G, U, true>
                            : sum_rows_kernel<I, DT, VEC, G, U, false>;
    k<<<grid, kTaskBlock, 0, s>>>(a);
  }
}

// Values per lane: 16 bytes, or what a narrower row has.
inline int sum_vec(int64_t F, int dtype) {
  if (F < 4) return 1;
  return dtype == TGX_DTYPE_F32 || F < 8 ? 4 : 8;
}

// Feature tiles of 64 lanes (the widest) that cover a row.
int sum_tiles(int64_t F, int dtype) {
  return static_cast<int>(ceil_div(F, int64_t{kWave} * sum_vec(F, dtype)));
}

template <typename I, int DT>
int sum_dispatch(const SumArgs<I, DT>& a, hipStream_t s) {
  const int64_t F = a.F;
  const int vec = sum_vec(F, DT);
  const int tiles = sum_tiles(F, DT);
  int lanes = 1;
  while (lanes < kWave && lanes < ceil_div(F, vec)) lanes *= 2;
  const auto with_vec = [&](auto vc) {
    constexpr int VEC = decltype(vc)::value;
    switch (lanes) {
      case 1: launch_sum<I, DT, VEC, 1>(a, tiles, s); break;
      case 2: launch_sum<I, DT, VEC, 2>(a, tiles, s); break;
      case 4: launch_sum<I, DT, VEC, 4>(a, tiles, s); break;
      default:
        // (Rows of fewer than 8 values have at most 4 lanes.)
        if constexpr (VEC == (DT == TGX_DTYPE_F32 ? 4 : 8)) {
          if (lanes == 8) launch_sum<I, DT, VEC, 8>(a, tiles, s);
          else if (lanes == 16) launch_sum<I, DT, VEC, 16>(a, tiles, s);
          else if (lanes == 32) launch_sum<I, DT, VEC, 32>(a, tiles, s);
          else launch_sum<I, DT, VEC, 64>(a, tiles, s);
        }
    }
  };
  if (vec == 1)
    with_vec(std::integral_constant<int, 1>{});
  else if (vec == 4)
    with_vec(std::integral_constant<int, 4>{});
  else if constexpr (DT != TGX_DTYPE_F32)
    with_vec(std::integral_constant<int, 8>{});
  TGX_LAUNCHED("sum_rows_kernel");
  if (a.plan.n_split > 0 && a.out) {
    sum_merge_kernel<DT><<<ceil_div(a.plan.n_split, kWavesPerBlock), kTaskBlock, 0, s>>>(
        a.plan, a.partial, a.out, F);
    TGX_LAUNCHED("sum_merge_kernel");
  }
  return TGX_OK;
}

// w_t[e'] = w[perm[e']]: the weights in transposed order, for launches that
// read them once per feature tile.
__global__ __launch_bounds__(kTaskBlock) void permute_weights_kernel(
    const float* __restrict__ w, const int32_t* __restrict__ perm, int64_t n,
    float* __restrict__ w_t) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kTaskBlock + threadIdx.x;
  if (e < n) w_t[e] = w[perm[e]];
}

// dw[perm[e']] = the feature tiles' sums for edge e', in tile order.
__global__ __launch_bounds__(kTaskBlock) void tile_dw_kernel(const float* __restrict__ part,
                                                             int tiles, int64_t n,
                                                             const int32_t* __restrict__ perm,
                                                             float* __restrict__ dw) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kTaskBlock + threadIdx.x;
  if (e >= n) return;
  float s = 0.f;
  for (int t = 0; t < tiles; ++t) s += part[t * n + e];
  dw[perm[e]] = s;
}

// dw for feature widths that span several tiles: one wave per edge group of
// the transposed CSR row, full-width dot product.
template <int DT>
__global__ __launch_bounds__(kTaskBlock) void sum_dw_wide_kernel(
    const int32_t* __restrict__ row_ptr_t, const int32_t* __restrict__ col_t,
    const int32_t* __restrict__ perm, const typename Elem<DT>::S* __restrict__ x,
    const typename Elem<DT>::S* __restrict__ dout, float* __restrict__ dw, int64_t n_src,
    int64_t F) {
  const int64_t j = global_wave();
  if (j >= n_src) return;
  const int64_t b = row_ptr_t[j], e = row_ptr_t[j + 1];
  for (int64_t k = b; k < e; ++k) {
    const int64_t i = col_t[k];
    float s = 0.f;
    for (int64_t f = lane_id(); f < F; f += kWave)
      s += Elem<DT>::load1(dout + i * F + f) * Elem<DT>::load1(x + j * F + f);
    s = group_sum<64>(s);
    if (lane_id() == 0) dw[perm[k]] = s;
  }
}

template <int V>
struct DtConst {
  static constexpr int value = V;
};
template <typename T>
struct IdxType {
  typedef T type;
};

// Calls f(DtConst<dtype>, IdxType<index type>) for a checked dtype code and
// index width.
template <typename F>
int with_types(int dtype, int idx_bits, F f) {
  if (dtype == TGX_DTYPE_BF16)
    return idx_bits == 32 ? f(DtConst<TGX_DTYPE_BF16>{}, IdxType<int32_t>{})
                          : f(DtConst<TGX_DTYPE_BF16>{}, IdxType<int64_t>{});
  if (dtype == TGX_DTYPE_F16)
    return idx_bits == 32 ? f(DtConst<TGX_DTYPE_F16>{}, IdxType<int32_t>{})
                          : f(DtConst<TGX_DTYPE_F16>{}, IdxType<int64_t>{});
  return idx_bits == 32 ? f(DtConst<TGX_DTYPE_F32>{}, IdxType<int32_t>{})
                        : f(DtConst<TGX_DTYPE_F32>{}, IdxType<int64_t>{});
}

}  // namespace

}  // namespace tgx

using namespace tgx;

extern "C" int tgx_partial_bytes(const tgx_row_plan* plan, int64_t state_floats,
                                 size_t* bytes) {
  TGX_REQUIRE(plan && bytes, "null pointer");
  TGX_REQUIRE(state_floats >= 0, "negative state size");
  *bytes = static_cast<size_t>(plan->n_chunks) * state_floats * sizeof(float);
  return TGX_OK;
}

extern "C" int tgx_csr_sum_fwd(const void* row_ptr, const void* col, int idx_bits,
                               const tgx_row_plan* plan, const void* x, const float* w,
                               void* out, int64_t n_dst, int64_t n_src, int64_t F, int dtype,
                               float* partial, void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(F > 0 && n_dst >= 0 && n_src >= 0, "bad sizes");
  if (dtype != TGX_DTYPE_F32 && dtype != TGX_DTYPE_BF16 && dtype != TGX_DTYPE_F16) {
    set_error("sum supports fp32, bf16 and fp16 features (dtype code %d)", dtype);
    return TGX_UNSUPPORTED;
  }
  int st = check_plan(plan, n_dst);
  if (st != TGX_OK) return st;
  if (n_dst == 0) return TGX_OK;
  TGX_REQUIRE(row_ptr && out && (x || n_src == 0), "null pointer");
  // A null col means the columns are the edge ids (x holds one row per edge).
  TGX_REQUIRE(col || n_src < (int64_t{1} << 31), "edge-id columns need fewer than 2^31 edges");
  // Gathered row indices are held in 32 bits.
  TGX_REQUIRE(n_src < (int64_t{1} << 31), "source tables need fewer than 2^31 rows");
  TGX_REQUIRE(plan->n_chunks == 0 || partial, "split rows need a partial buffer");
  hipStream_t s = as_stream(stream);
  TGX_PROFILE("csr_sum_fwd", s);
  auto run = [&](auto dt, auto idx) -> int {
    constexpr int DT = decltype(dt)::value;
    typedef typename decltype(idx)::type I;
    typedef typename Elem<DT>::S S;
    SumArgs<I, DT> a{static_cast<const I*>(row_ptr), static_cast<const I*>(col),
                     plan_view(*plan), static_cast<const S*>(x), w, nullptr,
                     static_cast<S*>(out), partial, nullptr, nullptr, nullptr, F, 0};
    return sum_dispatch(a, s);
  };
  return with_types(dtype, idx_bits, run);
}

// Workspace of a dw over several feature tiles: the tiles' dw and the weights
// in transposed order.  Past kSumWorkspaceMax dw runs as a pass of its own.
constexpr size_t kSumWorkspaceMax = size_t{2} << 30;

struct SumBwdLayout {
  int tiles;
  size_t part_off, w_off, bytes;
};

static SumBwdLayout sum_bwd_layout(int64_t n_edges, int64_t F, int dtype) {
  SumBwdLayout L{sum_tiles(F, dtype), 0, 0, 0};
  if (L.tiles > 1) {
    Carve c{nullptr, 0};
    L.part_off = reinterpret_cast<size_t>(c.take<float>(L.tiles * n_edges));
    L.w_off = reinterpret_cast<size_t>(c.take<float>(n_edges));
    L.bytes = align_up(c.used) <= kSumWorkspaceMax ? align_up(c.used) : 0;
  }
  return L;
}

extern "C" int tgx_csr_sum_bwd_workspace(int64_t n_edges, int64_t F, int dtype, size_t* bytes) {
  TGX_REQUIRE(bytes, "null bytes");
  TGX_REQUIRE(F > 0 && n_edges >= 0, "bad sizes");
  *bytes = sum_bwd_layout(n_edges, F, dtype).bytes;
  return TGX_OK;
}

extern "C" int tgx_csr_sum_bwd_ws(const int32_t* row_ptr_t, const int32_t* col_t,
                                  const int32_t* perm, const tgx_row_plan* plan_t,
                                  const void* x, const float* w, const void* dout, void* dx,
                                  float* dw, int64_t n_dst, int64_t n_src, int64_t n_edges,
                                  int64_t F, int dtype, float* partial, void* ws,
                                  size_t ws_bytes, void* stream) {
  TGX_REQUIRE(F > 0 && n_dst >= 0 && n_src >= 0 && n_edges >= 0, "bad sizes");
  if (dtype != TGX_DTYPE_F32 && dtype != TGX_DTYPE_BF16 && dtype != TGX_DTYPE_F16) {
    set_error("sum supports fp32, bf16 and fp16 features (dtype code %d)", dtype);
    return TGX_UNSUPPORTED;
  }
  int st = check_plan(plan_t, n_src);
  if (st != TGX_OK) return st;
  if (n_src == 0) return TGX_OK;
  TGX_REQUIRE(row_ptr_t && dout, "null pointer");
  // col_t / perm may be null for a graph without edges.
  TGX_REQUIRE(!dw || x, "dw needs x");
  TGX_REQUIRE(plan_t->n_chunks == 0 || partial || !dx, "split rows need a partial buffer");
  hipStream_t s = as_stream(stream);
  const SumBwdLayout L = sum_bwd_layout(n_edges, F, dtype);
  const bool tiled = L.bytes > 0 && ws && ws_bytes >= L.bytes && n_edges > 0;
  float* const part = tiled ? reinterpret_cast<float*>(static_cast<char*>(ws) + L.part_off)
                            : nullptr;
  TGX_PROFILE("csr_sum_bwd", s);
  auto run = [&](auto dt, auto) -> int {
    constexpr int DT = decltype(dt)::value;
    typedef typename Elem<DT>::S S;
    const S* xs = static_cast<const S*>(x);
    const S* gs = static_cast<const S*>(dout);
    const bool with_dw = dw && (L.tiles == 1 || tiled);   // dw from the sum's own pass
    if (dx || with_dw) {
      SumArgs<int32_t, DT> a{row_ptr_t, col_t, plan_view(*plan_t), gs, w, perm,
                             static_cast<S*>(dx), partial, nullptr, nullptr, nullptr, F, 0};
      if (tiled) {
        if (w) {
          float* w_t = reinterpret_cast<float*>(static_cast<char*>(ws) + L.w_off);
          permute_weights_kernel<<<ceil_div(n_edges, kTaskBlock), kTaskBlock, 0, s>>>(
              w, perm, n_edges, w_t);
          TGX_LAUNCHED("permute_weights_kernel");
          a.w = w_t;
        }
        a.wperm = nullptr;
      }
      if (with_dw) {
        a.self_x = xs;
        a.dw = tiled ? part : dw;
        a.dwperm = tiled ? nullptr : perm;
        a.dw_tile = tiled ? n_edges : 0;
      }
      const int r = sum_dispatch(a, s);
      if (r != TGX_OK) return r;
      if (tiled && with_dw) {
        tile_dw_kernel<<<ceil_div(n_edges, kTaskBlock), kTaskBlock, 0, s>>>(part, L.tiles, n_edges,
                                                                            perm, dw);
        TGX_LAUNCHED("tile_dw_kernel");
      }
    }
    if (dw && !with_dw) {
      sum_dw_wide_kernel<DT><<<ceil_div(n_src, kWavesPerBlock), kTaskBlock, 0, s>>>(
          row_ptr_t, col_t, perm, xs, gs, dw, n_src, F);
      TGX_LAUNCHED("sum_dw_wide_kernel");
    }
    return TGX_OK;
  };
  return with_types(dtype, 32, run);
}

extern "C" int tgx_csr_sum_bwd(const int32_t* row_ptr_t, const int32_t* col_t,
                               const int32_t* perm, const tgx_row_plan* plan_t,
                               const void* x, const float* w, const void* dout, void* dx,
                               float* dw, int64_t n_dst, int64_t n_src, int64_t F, int dtype,
                               float* partial, void* stream) {
  return tgx_csr_sum_bwd_ws(row_ptr_t, col_t, perm, plan_t, x, w, dout, dx, dw, n_dst, n_src, 0,
                            F, dtype, partial, nullptr, 0, stream);
}

extern "C" int tgx_csr_edge_dot(const void* row_ptr, const void* col, int idx_bits,
                                const tgx_row_plan* plan, const void* x, const void* dout,
                                float* dw, int64_t n_dst, int64_t n_src, int64_t F, int dtype,
                                void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(F > 0 && n_dst >= 0 && n_src >= 0, "bad sizes");
  if (dtype != TGX_DTYPE_F32 && dtype != TGX_DTYPE_BF16 && dtype != TGX_DTYPE_F16) {
    set_error("sum supports fp32, bf16 and fp16 features (dtype code %d)", dtype);
    return TGX_UNSUPPORTED;
  }
  if (F > 32) {
    set_error("tgx_csr_edge_dot covers F <= 32 (got %lld); wider rows take the dw output "
              "of tgx_csr_sum_bwd", static_cast<long long>(F));
    return TGX_UNSUPPORTED;
  }
  int st = check_plan(plan, n_dst);
  if (st != TGX_OK) return st;
  if (n_dst == 0) return TGX_OK;
  TGX_REQUIRE(row_ptr && col && x && dout && dw, "null pointer");
  TGX_REQUIRE(n_src < (int64_t{1} << 31), "source tables need fewer than 2^31 rows");
  hipStream_t s = as_stream(stream);
  TGX_PROFILE("csr_edge_dot", s);
  auto run = [&](auto dt, auto idx) -> int {
    constexpr int DT = decltype(dt)::value;
    typedef typename decltype(idx)::type I;
    typedef typename Elem<DT>::S S;
    // The sum kernel over the CSR with the row's own dout as `self`: it
    // writes dw[e] = <dout[i], x[col[e]]> in edge order and no sums.
    SumArgs<I, DT> a{static_cast<const I*>(row_ptr), static_cast<const I*>(col),
                     plan_view(*plan), static_cast<const S*>(x), nullptr, nullptr, nullptr,
                     nullptr, static_cast<const S*>(dout), dw, nullptr, F, 0};
    return sum_dispatch(a, s);
  };
  return with_types(dtype, idx_bits, run);
}

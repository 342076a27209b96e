// Edge networks of two Linear layers whose first layer reads destination fields:
//   score_e = w2 . act(W1 [x_src[j] | x_dst[i] | field_e] + b1) + b2.
// The first layer is linear in each field, so its destination columns are
// applied once per row instead of once per edge, pt[i] = W1_dst x_dst[i] + b1, and
//   z_e = pt[i] + W1_src x_src[j] + W1_edge field_e.
// (The source columns stay with the edge: a gathered row of W1_src x_src would
// be another random line per edge, and those bound the pass: 4M edges, 19-16-1,
// backward 245 us with them gathered, 223 so.)
// The reference evaluates the concatenation per edge (python/tiga/compiler/
// edge_nn_attention.py:127-338; its VJP :344-611), as the edge-MLP kernels of
// tgx_nn.hip do, which take every other chain.
//
// Backward of the online-softmax attention over the scores (the logsumexp
// recompute form of tgx_edge_mlp_attention_backward), one pass over the edges:
// z is formed again, dz_e = ds_e w2 act'(z); a wave stages its 64 edges' dz in
// LDS and from there
//   - sums dz over each destination row's edges (edges are in row order, so a
//     row is a run of lanes); rows that cross waves leave partial sums that
//     the row pass adds in order.  No per-edge gradient of a destination field
//     goes to memory: dx_dst[i] = W1_dst^T (sum dz) and dW1_dst = sum_i
//     (sum dz) (x) x_dst[i] come from the row pass;
//   - feeds fp32 MFMA (exact fp32 products and sums) with dz (x) [x_src |
//     field_e | 1], the other columns of dW1 and db1.
// Source and edge fields get per-edge gradient rows W1^T dz (the folded value
// gradient alpha dout[i] added), as tgx_edge_mlp_attention_backward writes.
// Every sum has a fixed order.
//
// 131,072 nodes, 3.9M edges, 19-16-1, leaky ReLU, value 8 folded (MI355X):
// scores 63 us, backward 214, rows and weights 35; forward and backward of the
// layer, with the softmax and the transposed sum, 447 us (630 on the edge-MLP
// kernels).  The edge pass is bound by the gathered lines (about 73 us of it) and
// by the exposed latency of its chain of loads, weights and LDS sums at four
// waves a SIMD: with a third fewer instructions (arguments read from the
// argument segment instead of spilled) it took 214 us against 224.
#include <hip/hip_runtime.h>

#include "tgx_nn_common.h"
#include "tgx_profile.h"

namespace tgx {
namespace {

using namespace mlp;

// Columns of an edge's input row u: source fields, edge fields, and 1 (the
// bias); of a destination's: its fields.
constexpr int kU = 16, kSrcCols = 8, kEdgeCols = 7;
// Hidden units, padded: one tile of the MFMA.
constexpr int HP = 16;

// The fields of one role: at most kRoleSegs, columns from 0 in the role.
constexpr int kRoleSegs = 2;
struct Field {
  const float* ptr;
  float* grad;        // [E, width] (destination fields: [n_dst, width])
  int64_t stride;     // floats between rows
  int width, off;     // columns off .. off + width of the role
  int col;            // first column of W1
};
struct Role {
  Field f[kRoleSegs];
  int n, width;
};

struct ProjView {
  Role src, dst, edge;
  int in_width, hidden, act;
  float param, param2;
  int W;                    // padded width of the caller's weight-gradient blocks
  const float *w1, *b1, *w2, *b2;   // [hidden, in_width], [hidden], [hidden], [1]; biases or null
  // State (floats): pt [n_dst, HP], the packed weights (Packed), and
  // [n_dst] for near_kink.
  float *pt, *packed, *bound;
  Field in[kMaxSegments];   // the fields in input order
  int n_in, in_role[kMaxSegments];
  // Backward: each row's logsumexp, output and its gradient, the value rows,
  // the source field that takes the value's gradient (or -1).
  const float *lse, *out, *dout, *value;
  int value_width, fold;
};

// Offsets of the packed weights: W1's source and edge columns and, at wt, its
// destination columns, both as [column][HP] (a column is one scalar load), the
// second layer, b1, b2, the largest |W1| of each column of both and |b1|.
struct Packed {
  static constexpr int wt = HP * kU, w2 = 2 * HP * kU, b1 = w2 + HP, b2 = b1 + HP, most = b2 + 1,
                       end = most + 2 * kU + 1;
};
// b1 of the units past `hidden`, whose other weights are 0: far from any kink.
constexpr float kNoUnit = 1e30f;

// x[c] of a role's fields at `row`, 0 past their columns.  A single field's loads
// are all in flight at once; a second one's, into the same registers, wait for
// the first's.
template <int N>
__device__ __forceinline__ void gather_role(const Role& r, int64_t row, float (&x)[N]) {
  const int w0 = r.f[0].width;
  const float* p = r.f[0].ptr + row * r.f[0].stride;
#pragma unroll
  for (int b = 0; b < N; b += 4) {
    if (b + 4 <= w0) {
#pragma unroll
      for (int c = b; c < b + 4; ++c) x[c] = p[c];
    } else if (b < w0) {
#pragma unroll
      for (int c = b; c < b + 4; ++c) {
        const float y = p[c < w0 ? c : b];
        x[c] = c < w0 ? y : 0.f;
      }
    } else {
#pragma unroll
      for (int c = b; c < b + 4; ++c) x[c] = 0.f;
    }
  }
  if (r.n > 1) {
    const int off = r.f[1].off, end = off + r.f[1].width;
    p = r.f[1].ptr + row * r.f[1].stride - off;
#pragma unroll
    for (int c = 0; c < N; ++c)
      if (c >= off && c < end) x[c] = p[c];
  }
}

// g to the fields' gradient rows of edge e; field `fold` (when >= 0) also
// receives alpha d, d the value's row gradient.
template <int N>
__device__ __forceinline__ void scatter_role(const Role& r, int64_t e, const float (&g)[N],
                                             int fold = -1, float alpha = 0.f,
                                             const float* d = nullptr) {
#pragma unroll
  for (int s = 0; s < kRoleSegs; ++s) {
    if (s >= r.n) break;
    const int off = r.f[s].off, end = off + r.f[s].width;
    float* p = r.f[s].grad + e * r.f[s].width - off;
    const bool add = s == fold;
#pragma unroll
    for (int b = 0; b < N; b += 4) {
      if (b + 4 > off && b < end) {
        float x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = g[b + c];
        if (b >= off && b + 4 <= end) {
          if (add)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[c] = fmaf(alpha, d[b + c - off], x[c]);
#pragma unroll
          for (int c = 0; c < 4; ++c) p[b + c] = x[c];
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (b + c >= off && b + c < end)
              p[b + c] = add ? fmaf(alpha, d[b + c - off], x[c]) : x[c];
        }
      }
    }
  }
}

__device__ __forceinline__ int w1_column(const Role& r, int c) {
  for (int s = 0; s < r.n; ++s)
    if (c >= r.f[s].off && c < r.f[s].off + r.f[s].width) return r.f[s].col + c - r.f[s].off;
  return -1;
}

__global__ __launch_bounds__(256) void pack_weights_kernel(ProjView v) {
  typedef Packed P;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P::end) return;
  const auto column = [&](bool to_dst, int c) {
    return to_dst ? w1_column(v.dst, c)
           : c < kSrcCols ? w1_column(v.src, c) : w1_column(v.edge, c - kSrcCols);
  };
  float x = 0.f;
  if (i < P::w2) {
    const int h = i % HP, k = column(i >= P::wt, i / HP % kU);
    if (h < v.hidden && k >= 0) x = v.w1[h * v.in_width + k];
  } else if (i < P::b1) {
    if (i - P::w2 < v.hidden) x = v.w2[i - P::w2];
  } else if (i < P::b2) {
    const int h = i - P::b1;
    x = h >= v.hidden ? kNoUnit : v.b1 ? v.b1[h] : 0.f;
  } else if (i < P::most) {
    if (v.b2) x = v.b2[0];
  } else {
    const int c = i - P::most;
    const int k = c < 2 * kU ? column(c >= kU, c % kU) : -1;
    for (int h = 0; h < v.hidden; ++h) {
      if (k >= 0) x = fmaxf(x, fabsf(v.w1[h * v.in_width + k]));
      if (c == 2 * kU && v.b1) x = fmaxf(x, fabsf(v.b1[h]));
    }
  }
  v.packed[i] = x;
}

// pt, a thread per node, the weights in scalar registers.
__global__ __launch_bounds__(256) void project_nodes_kernel(ProjView v, int64_t n_dst) {
  typedef Packed P;
  cfloat* wu = scalar_weights(v.packed);
  const int64_t n = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (n >= n_dst) return;
  float x[kU], z[HP], m = wu[P::most + 2 * kU];
  gather_role<kU>(v.dst, n, x);
#pragma unroll
  for (int h = 0; h < HP; ++h) z[h] = wu[P::b1 + h];
#pragma unroll
  for (int c = 0; c < kU; ++c) {
    if (c < v.dst.width) {
      m = fmaf(wu[P::most + kU + c], fabsf(x[c]), m);
#pragma unroll
      for (int h = 0; h < HP; ++h) z[h] = fmaf(wu[P::wt + c * HP + h], x[c], z[h]);
    }
  }
#pragma unroll
  for (int h = 0; h < HP; h += 4)
    *reinterpret_cast<f32x4*>(v.pt + n * HP + h) = f32x4{z[h], z[h + 1], z[h + 2], z[h + 3]};
  v.bound[n] = m;
}

// z of an edge: its destination's row of pt, then its source fields (xs) and its
// own (ed), both 0 past their columns.
__device__ __forceinline__ void edge_z(const ProjView& v, cfloat* wu, int64_t i,
                                       const float (&xs)[kSrcCols], const float (&ed)[8],
                                       float (&z)[HP]) {
  const f32x4* d = reinterpret_cast<const f32x4*>(v.pt + i * HP);
#pragma unroll
  for (int k = 0; k < HP / 4; ++k) {
    const f32x4 x = d[k];
#pragma unroll
    for (int r = 0; r < 4; ++r) z[4 * k + r] = x[r];
  }
#pragma unroll
  for (int b = 0; b < kSrcCols; b += 4) {
    if (b < v.src.width) {
#pragma unroll
      for (int c = b; c < b + 4; ++c)
#pragma unroll
        for (int h = 0; h < HP; ++h) z[h] = fmaf(wu[c * HP + h], xs[c], z[h]);
    }
  }
#pragma unroll
  for (int c = 0; c < kEdgeCols; ++c) {
    if (c < v.edge.width) {
#pragma unroll
      for (int h = 0; h < HP; ++h) z[h] = fmaf(wu[(kSrcCols + c) * HP + h], ed[c], z[h]);
    }
  }
}

__device__ __forceinline__ float edge_score(cfloat* wu, const float (&a)[HP]) {
  cfloat* w2 = wu + Packed::w2;
  float s = wu[Packed::b2];
#pragma unroll
  for (int h = 0; h < HP; ++h) s = fmaf(w2[h], a[h], s);
  return s;
}

// Whether rounding may decide on which side of 0 some unit of the edge lies, and
// so, where the activation has a kink there, its derivative: z as sums per node
// and z summed over the concatenated inputs are each within 33 roundings of
// |b1| + sum |w x| of the exact value, that is 2^-18 of it apart together; twice that is
// asked, with each column's largest weight.  `bound` has the destination's part.
__device__ __forceinline__ bool near_kink(cfloat* wu, const float (&xs)[kSrcCols],
                                          const float (&ed)[8], const float (&z)[HP],
                                          float bound) {
  cfloat* most = wu + Packed::most;
#pragma unroll
  for (int c = 0; c < kSrcCols; ++c) bound = fmaf(most[c], fabsf(xs[c]), bound);
#pragma unroll
  for (int c = 0; c < kEdgeCols; ++c) bound = fmaf(most[kSrcCols + c], fabsf(ed[c]), bound);
  float least = fabsf(z[0]);
#pragma unroll
  for (int h = 1; h < HP; ++h) least = fminf(least, fabsf(z[h]));
  return least <= bound * 0x1p-17f;
}

// z summed over the concatenated inputs in their order, as the edge-MLP kernels
// do: which side of the kink an edge is on does not depend on the route.
__device__ __forceinline__ void direct_z(const ProjView& v, cfloat* wu, int64_t e, int64_t j,
                                         int64_t i, float (&z)[HP]) {
  typedef Packed P;
#pragma unroll
  for (int h = 0; h < HP; ++h) z[h] = wu[P::b1 + h];
#pragma unroll
  for (int s = 0; s < kMaxSegments; ++s) {
    if (s >= v.n_in) break;
    const int64_t row = v.in_role[s] == TGX_ROLE_SRC ? j : v.in_role[s] == TGX_ROLE_DST ? i : e;
    const float* p = v.in[s].ptr + row * v.in[s].stride;
    const int first = v.in_role[s] == TGX_ROLE_SRC   ? 0
                      : v.in_role[s] == TGX_ROLE_DST ? P::wt
                                                     : kSrcCols * HP;
#pragma unroll 1
    for (int c0 = 0; c0 < v.in[s].width; c0 += 4) {
      cfloat* w = wu + first + (v.in[s].off + c0) * HP;
      float x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] = c0 + c < v.in[s].width ? p[c0 + c] : 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c0 + c < v.in[s].width)
#pragma unroll
          for (int h = 0; h < HP; ++h) z[h] = fmaf(w[c * HP + h], x[c], z[h]);
    }
  }
}

// ds of an edge and its weight alpha, from its score (attention_score_grad of
// the edge-MLP kernels).
__device__ __forceinline__ float score_grad(const ProjView& v, int64_t i, int64_t j, float s,
                                            const float (&xs)[kSrcCols], float& alpha) {
  alpha = __expf(s - v.lse[i]);
  const int F = v.value_width;
  const float* d = v.dout + i * F;
  const float* o = v.out + i * F;
  const float* x = v.value + j * F;
  float dv = 0.f, dd = 0.f;
  if ((F & 3) == 0 && v.fold == 0 && v.src.n == 1) {   // the value row is xs
#pragma unroll
    for (int f = 0; f < kSrcCols; f += 4) {
      if (f < F) {
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(d + f);
        const f32x4 o4 = *reinterpret_cast<const f32x4*>(o + f);
        dv += d4[0] * xs[f] + d4[1] * xs[f + 1] + d4[2] * xs[f + 2] + d4[3] * xs[f + 3];
        dd += d4[0] * o4[0] + d4[1] * o4[1] + d4[2] * o4[2] + d4[3] * o4[3];
      }
    }
  } else if ((F & 3) == 0) {
    for (int f = 0; f < F; f += 4) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(d + f);
      const f32x4 x4 = *reinterpret_cast<const f32x4*>(x + f);
      const f32x4 o4 = *reinterpret_cast<const f32x4*>(o + f);
      dv += d4[0] * x4[0] + d4[1] * x4[1] + d4[2] * x4[2] + d4[3] * x4[3];
      dd += d4[0] * o4[0] + d4[1] * o4[1] + d4[2] * o4[2] + d4[3] * o4[3];
    }
  } else {
    for (int f = 0; f < F; ++f) {
      dv += d[f] * x[f];
      dd += d[f] * o[f];
    }
  }
  return alpha * (dv - dd);
}

// A thread per edge, bound by the gathered line of the source row (two edges
// per thread, to share the weights' scalar loads: 67.8 us against 64.4).
template <typename I, int ACT>
__global__ __launch_bounds__(256) void projected_scores_kernel(const I* __restrict__ col,
                                                               const int32_t* __restrict__ dst,
                                                               int64_t n_edges, ProjView v,
                                                               float* __restrict__ scores) {
  cfloat* wu = scalar_weights(v.packed);
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n_edges) return;
  float ed[8], xs[kSrcCols], z[HP], a[HP];
  const int64_t j = col[e], i = dst[e];
  gather_role<8>(v.edge, e, ed);
  gather_role<kSrcCols>(v.src, j, xs);
  edge_z(v, wu, i, xs, ed, z);
  activate_all<HP>(z, a, ACT >= 0 ? ACT : v.act, v.param, v.param2, (v.hidden + 3) / 4,
                   v.hidden);
  scores[e] = edge_score(wu, a);
}

typedef float f32x4m __attribute__((ext_vector_type(4)));

// The shape fields, hidden from the optimizer: what is derived from them is
// formed where it is used (the columns' guards, hoisted out of the loop, would
// take scalar registers that spill: 226 against 167 spills).
__device__ __forceinline__ void launder(Role& r) {
  asm volatile("" : "+s"(r.n), "+s"(r.width));
#pragma unroll
  for (int s = 0; s < kRoleSegs; ++s)
    asm volatile("" : "+s"(r.f[s].width), "+s"(r.f[s].off), "+s"(r.f[s].stride));
}

// The pass over the edges, a thread per edge and 64 consecutive edges per wave.
// A row's sum of dz goes to dzt where one wave saw all its edges, else to part,
// two slots of HP per wave: 0 the run that continues a row from before the
// wave, 1 the run that leaves it unfinished.
template <typename I, int ACT>
__global__ __launch_bounds__(256, ACT < 0 ? 3 : 4) void projected_bwd_kernel(
    const I* __restrict__ col, const int32_t* __restrict__ dst, int64_t n_edges, int64_t chunk,
    ProjView v_arg, float* __restrict__ dzt,
    float* __restrict__ part, float* __restrict__ sums) {
  // (Rows of 16: a wave's reads below are of consecutive words, its 16-byte
  // writes two lanes to a bank.)
  constexpr int LG = HP, LU = kU;
  __shared__ alignas(16) float g_stage[4][kWave * LG];
  __shared__ alignas(16) float u_stage[4][kWave * LU];
  __shared__ int seg_first[4][kWave + 1], seg_row[4][kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int q = lane >> 4, hh = lane & 15;
  float* const gs = g_stage[wave];
  float* const us = u_stage[wave];
  cfloat* const w_all = scalar_weights(v_arg.packed);
  f32x4m acc{0.f, 0.f, 0.f, 0.f};
  float last_w[HP], last_b = 0.f;
#pragma unroll
  for (int h = 0; h < HP; ++h) last_w[h] = 0.f;
  const int64_t e0 = static_cast<int64_t>(blockIdx.x) * chunk;
  const int64_t e1 = e0 + chunk < n_edges ? e0 + chunk : n_edges;
  for (int64_t base = e0; base < e1; base += 256) {
    // (Weights are re-read in every step, scalar-cache hits: hoisted out of
    // the loop they would all be live at once.)
    cfloat* wu = opaque(w_all);
    ProjView v = v_arg;
    launder(v.src);
    launder(v.edge);
    const int64_t wave_base = base + kWave * wave;
    const int64_t e = wave_base + lane;
    const bool valid = e < e1;
    const int nv = static_cast<int>(wave_base >= e1 ? 0 : e1 - wave_base < kWave ? e1 - wave_base
                                                                               : kWave);
    const int64_t ec = valid ? e : e0;
    const int64_t j = col[ec], i = dst[ec];
    // The rows on both sides of the wave's edges.
    const int row_before = wave_base > 0 && wave_base < e1 ? dst[wave_base - 1] : -1;
    const int row_after = wave_base + kWave < n_edges ? dst[wave_base + kWave] : -1;
    float ed[8], xs[kSrcCols], z[HP], dz[HP];
    gather_role<8>(v.edge, ec, ed);
    gather_role<kSrcCols>(v.src, j, xs);
    edge_z(v, wu, i, xs, ed, z);
    if (__any(near_kink(wu, xs, ed, z, v.bound[i]))) direct_z(v, wu, ec, j, i, z);
    const int nb = (v.hidden + 3) / 4;
    float alpha;
    {
      float a[HP];
      activate_all<HP>(z, a, ACT >= 0 ? ACT : v.act, v.param, v.param2, nb, v.hidden);
      const float s = edge_score(wu, a);
      float ds = score_grad(v, i, j, s, xs, alpha);
      if (!valid) {
        ds = 0.f;
        alpha = 0.f;
      }
      last_b += ds;
      cfloat* w2 = wu + Packed::w2;
      float g[HP];
#pragma unroll
      for (int h = 0; h < HP; ++h) {
        // (A lane past the range holds another edge's values: its terms are
        // selected away, not multiplied by 0.)
        last_w[h] += valid ? ds * a[h] : 0.f;
        g[h] = ds * w2[h];
      }
      activate_grad_all<HP>(z, g, dz, ACT >= 0 ? ACT : v.act, v.param, v.param2, nb, v.hidden);
    }
#pragma unroll
    for (int h = 0; h < HP; h += 4)
      *reinterpret_cast<f32x4*>(gs + lane * LG + h) =
          valid ? f32x4{dz[h], dz[h + 1], dz[h + 2], dz[h + 3]} : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < kU; c += 4) {
      f32x4 u;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        u[k] = !valid ? 0.f : c + k < kSrcCols ? xs[(c + k) % kSrcCols]
               : c + k < kU - 1 ? ed[(c + k) % kSrcCols] : 1.f;
      *reinterpret_cast<f32x4*>(us + lane * LU + c) = u;
    }
    // Runs of lanes with one destination row.
    const int row = static_cast<int>(i);
    const int before = __shfl_up(row, 1, kWave);
    const bool head = valid && (lane == 0 || row != before);
    const uint64_t heads = __ballot(head);
    const int n_seg = __popcll(heads);
    const bool continued = row_before == __builtin_amdgcn_readlane(row, 0);
    const bool unfinished = row_after == __builtin_amdgcn_readlane(row, kWave - 1);
    if (head) {
      const int k = __popcll(heads & (lane == 0 ? 0ull : (~0ull >> (kWave - lane))));
      seg_first[wave][k] = lane;
      seg_row[wave][k] = row;
    }
    if (lane == 0) seg_first[wave][n_seg] = nv;
    // The edge's own gradient rows.
    {
      float gx[kSrcCols], ge[8];
#pragma unroll
      for (int c = 0; c < kSrcCols; ++c) gx[c] = 0.f;
#pragma unroll
      for (int c = 0; c < 8; ++c) ge[c] = 0.f;
#pragma unroll
      for (int c = 0; c < kSrcCols; c += 4) {
        if (c < v.src.width) {
#pragma unroll
          for (int h = 0; h < HP; ++h)
#pragma unroll
            for (int k = c; k < c + 4; ++k) gx[k] = fmaf(wu[k * HP + h], dz[h], gx[k]);
        }
        if (c < v.edge.width) {
#pragma unroll
          for (int h = 0; h < HP; ++h)
#pragma unroll
            for (int k = c; k < c + 4 && k < kEdgeCols; ++k)
              ge[k] = fmaf(wu[(kSrcCols + k) * HP + h], dz[h], ge[k]);
        }
      }
      if (valid) {
        scatter_role<kSrcCols>(v.src, e, gx, v.fold, alpha, v.dout + i * v.value_width);
        scatter_role<8>(v.edge, e, ge);
      }
    }
    // One wave's LDS accesses complete in issue order.
    __builtin_amdgcn_wave_barrier();
    // Row sums: few runs are summed by all four 16-lane groups, many by one
    // group each.
    auto store_sum = [&](int k, float s) TGX_INLINE_LAMBDA {
      float* const slots = part + (wave_base / kWave) * 2 * HP;
      float* p = k == 0 && continued            ? slots
                 : k == n_seg - 1 && unfinished ? slots + HP
                                                : dzt + static_cast<int64_t>(seg_row[wave][k]) * HP;
      p[hh] = s;
    };
    if (n_seg < 4) {
      for (int k = 0; k < n_seg; ++k) {
        const int x1 = seg_first[wave][k + 1];
        float s = 0.f;
        for (int x = seg_first[wave][k] + q; x < x1; x += 4) s += gs[x * LG + hh];
        s += __shfl_xor(s, 16, kWave);
        s += __shfl_xor(s, 32, kWave);
        if (q == 0) store_sum(k, s);
      }
    } else {
      for (int k = q; k < n_seg; k += 4) {
        const int x1 = seg_first[wave][k + 1];
        float s = 0.f;
        for (int x = seg_first[wave][k]; x < x1; ++x) s += gs[x * LG + hh];
        store_sum(k, s);
      }
    }
    // dz (x) u over the wave's edges: A[h = l % 16][edge l / 16],
    // B[edge l / 16][column l % 16].
#pragma unroll
    for (int x = 0; x < kWave; x += 4)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(gs[(x + q) * LG + hh], us[(x + q) * LU + hh],
                                                 acc, 0, 0, 0);
    __builtin_amdgcn_wave_barrier();
  }
  // The block's sums: per wave into LDS, then the four waves in order.
  __syncthreads();
  constexpr int N = HP * (kU + 1) + 1;
  static_assert(N <= kWave * LG, "a wave's sums fit its staging");
#pragma unroll
  for (int h = 0; h < HP; ++h) gs[lane * LG + h] = last_w[h];
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) last_b += __shfl_xor(last_b, m, kWave);
  __builtin_amdgcn_wave_barrier();
  float lw = 0.f;
  for (int x = q; x < kWave; x += 4) lw += gs[x * LG + hh];
  lw += __shfl_xor(lw, 16, kWave);
  lw += __shfl_xor(lw, 32, kWave);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int r = 0; r < 4; ++r) gs[(4 * q + r) * kU + hh] = acc[r];
  if (q == 0) gs[HP * kU + hh] = lw;
  if (lane == 0) gs[HP * (kU + 1)] = last_b;
  __syncthreads();
  for (int c = threadIdx.x; c < N; c += 256) {
    const float s = ((g_stage[0][c] + g_stage[1][c]) + g_stage[2][c]) + g_stage[3][c];
    sums[static_cast<int64_t>(c) * gridDim.x + blockIdx.x] = s;
  }
}

// Destination rows: the sum of dz (partial sums added in edge order), its
// fields' gradient W1_dst^T (sum dz), and the sums (sum dz) (x) x_dst on MFMA.
// A 16-lane group per row, lane hh holding hidden unit hh.  A row over more than
// kOwnPartials waves of edges is summed by the workgroup's 16 groups, every 16th
// partial sum each (a hub of a million edges has 16,000: backward 3.57 ms with
// one group walking them, 0.23 so).
constexpr int kRowGroups = 16, kOwnPartials = 16;
template <typename I>
__global__ __launch_bounds__(256) void projected_rows_kernel(const I* __restrict__ row_ptr,
                                                             int64_t n_rows, ProjView v,
                                                             const float* __restrict__ dzt,
                                                             const float* __restrict__ part,
                                                             float* __restrict__ sums) {
  __shared__ float red[4][HP * kU];
  __shared__ int range[kRowGroups][2];
  __shared__ float fold[kRowGroups][HP];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int q = lane >> 4, hh = lane & 15;
  const int group = threadIdx.x >> 4;
  float wt[HP];   // column hh of W1_dst
#pragma unroll
  for (int h = 0; h < HP; ++h) wt[h] = v.packed[Packed::wt + hh * HP + h];
  // The destination field that column hh belongs to.
  const float* x = nullptr;
  float* grad = nullptr;
  int64_t stride = 0;
  int width = 0;
#pragma unroll
  for (int s = 0; s < kRoleSegs; ++s)
    if (s < v.dst.n && hh >= v.dst.f[s].off && hh < v.dst.f[s].off + v.dst.f[s].width) {
      x = v.dst.f[s].ptr + hh - v.dst.f[s].off;
      stride = v.dst.f[s].stride;
      width = v.dst.f[s].width;
      grad = v.dst.f[s].grad + hh - v.dst.f[s].off;
    }
  f32x4m acc{0.f, 0.f, 0.f, 0.f};
  const int64_t step = static_cast<int64_t>(gridDim.x) * kRowGroups;
  for (int64_t first = static_cast<int64_t>(blockIdx.x) * kRowGroups; first < n_rows;
       first += step) {
    const int64_t row = first + group;
    const bool valid = row < n_rows;
    const int64_t r0 = valid ? row_ptr[row] : 0, r1 = valid ? row_ptr[row + 1] : 0;
    // A row without edges has no part in the layer: its fields are not read
    // (they may be Inf or NaN, a mean over no neighbours) and its gradient is 0.
    const bool any = r1 > r0;
    const int64_t w0 = r0 / kWave, w1 = any ? (r1 - 1) / kWave : w0;
    const bool shared = w1 - w0 > kOwnPartials;
    float dz = 0.f, u = 0.f;
    if (any) {
      if (w0 == w1) {
        dz = dzt[row * HP + hh];
      } else if (!shared) {
        dz = part[(w0 * 2 + 1) * HP + hh];
        for (int64_t w = w0 + 1; w <= w1; ++w) dz += part[w * 2 * HP + hh];
      }
      if (x) u = x[row * stride];
    }
    if (__syncthreads_or(shared)) {
      if (hh == 0) {   // (Below 2^31 edges: a wave's index fits.)
        range[group][0] = static_cast<int>(w0);
        range[group][1] = static_cast<int>(shared ? w1 : w0);
      }
      __syncthreads();
      for (int k = 0; k < kRowGroups; ++k) {
        const int64_t a = range[k][0], b = range[k][1];
        if (a == b) continue;
        float s = group == 0 ? part[(a * 2 + 1) * HP + hh] : 0.f;
        int64_t w = a + 1 + group;
        for (; w + 7 * kRowGroups <= b; w += 8 * kRowGroups) {
          float y[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) y[r] = part[(w + r * kRowGroups) * 2 * HP + hh];
#pragma unroll
          for (int r = 0; r < 8; ++r) s += y[r];
        }
        for (; w <= b; w += kRowGroups) s += part[w * 2 * HP + hh];
        fold[group][hh] = s;
        __syncthreads();
        if (group == k)
          for (int r = 0; r < kRowGroups; ++r) dz += fold[r][hh];
        __syncthreads();
      }
    }
    float g = 0.f;
#pragma unroll
    for (int h = 0; h < HP; ++h) g = fmaf(wt[h], __shfl(dz, 16 * q + h, kWave), g);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(dz, u, acc, 0, 0, 0);
    if (valid && x) grad[row * width] = any ? g : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][(4 * q + r) * kU + hh] = acc[r];
  __syncthreads();
  for (int c = threadIdx.x; c < HP * kU; c += 256)
    sums[static_cast<int64_t>(c) * gridDim.x + blockIdx.x] =
        ((red[0][c] + red[1][c]) + red[2][c]) + red[3][c];
}

// The weight-gradient blocks [W*W | W] of both layers: one wave per element,
// the blocks' sums added in a fixed order; padding gets 0.
__global__ __launch_bounds__(256) void projected_weights_kernel(ProjView v,
                                                                const float* __restrict__ edge_sums,
                                                                int edge_blocks,
                                                                const float* __restrict__ row_sums,
                                                                int row_blocks,
                                                                float* __restrict__ dweights) {
  const int W = v.W, nw = W * W + W;
  const int x = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (x >= 2 * nw) return;
  const int l = x / nw, y = x % nw;
  const float* p = nullptr;
  int n = 0;
  if (l == 0) {
    const bool bias = y >= W * W;
    const int h = bias ? y - W * W : y / W, k = bias ? -1 : y % W;
    int c = bias ? kU - 1 : -1;
    bool rows = false;
    if (!bias) {
      const auto column = [&](const Role& r) {
        for (int s = 0; s < r.n; ++s)
          if (k >= r.f[s].col && k < r.f[s].col + r.f[s].width) return r.f[s].off + k - r.f[s].col;
        return -1;
      };
      c = column(v.src);
      if (c < 0 && column(v.edge) >= 0) c = kSrcCols + column(v.edge);
      if (c < 0) {
        c = column(v.dst);
        rows = c >= 0;
      }
    }
    if (h < v.hidden && c >= 0) {
      n = rows ? row_blocks : edge_blocks;
      p = (rows ? row_sums : edge_sums) + static_cast<int64_t>(h * kU + c) * n;
    }
  } else if (y < W ? y < v.hidden : y == W * W) {
    n = edge_blocks;
    p = edge_sums + static_cast<int64_t>(y < W ? HP * kU + y : HP * (kU + 1)) * n;
  }
  float s = 0.f;
  for (int b = lane; b < n; b += kWave) s += p[b];
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) s += __shfl_xor(s, m, kWave);
  if (lane == 0) dweights[x] = s;
}

// Whether the kernels cover the chain, and its view (state pointers unset).
int proj_view(const tgx_edge_mlp* m, ProjView* out) {
  TGX_REQUIRE(m, "null mlp");
  ProjView v{};
  const auto unsupported = [](const char* what) {
    set_error("projected edge networks cover %s", what);
    return TGX_UNSUPPORTED;
  };
  if (m->n_layers != 2 || m->width > 32 || uses_math_tier(m))
    return unsupported("two layers of up to 32, without LayerNorm or the second function set");
  // (direct_z minds a kink at 0; these have theirs elsewhere.)
  if (m->act[0] < TGX_ACT_IDENTITY || m->act[0] > TGX_ACT_HARDSWISH ||
      m->act[0] == TGX_ACT_HARDTANH || m->act[0] == TGX_ACT_HARDSIGMOID ||
      m->act[0] == TGX_ACT_HARDSWISH)
    return unsupported("the first set of functions without the clamped ones");
  // (Every other function is finite at kNoUnit; a softplus whose threshold lies
  // beyond it takes the exponential there.)
  if (m->act[0] == TGX_ACT_SOFTPLUS && m->act_param[0] > 0.f &&
      !(m->act_param[0] * kNoUnit > m->act_param2[0]))
    return unsupported("softplus with a threshold below 1e30 beta");
  TGX_REQUIRE(m->width == 16 || m->width == 24 || m->width == 32, "bad padded width");
  TGX_REQUIRE(m->n_segments >= 1 && m->n_segments <= kMaxSegments, "bad segment count");
  v.hidden = m->out_width[0] ? m->out_width[0] : m->width;
  TGX_REQUIRE(v.hidden >= 1 && v.hidden <= m->width, "bad hidden width");
  TGX_REQUIRE(m->out_width[1] == 0 || m->out_width[1] == 1, "the last layer has one output");
  // (Two tiles, 17 to 32 units, padded more and held more than they saved: forward
  // and backward of 3.7M edges, hidden 20 leaky 620 us against 630 of the edge-MLP
  // kernels, 24 ReLU 671 against 603, 32 GELU of 2.1M edges 749 against 587.  One
  // tile, 3.7M edges: leaky 8 331 against 390, SiLU 503 against 640, GELU 555
  // against 677.)
  if (v.hidden > HP) return unsupported("up to 16 hidden units");
  v.act = m->act[0];
  v.param = m->act_param[0];
  v.param2 = m->act_param2[0];
  v.W = m->width;
  Role* const roles[3] = {&v.src, &v.dst, &v.edge};
  int k = 0;
  for (int s = 0; s < m->n_segments; ++s) {
    const int role = m->seg_role[s];
    TGX_REQUIRE(role >= TGX_ROLE_SRC && role <= TGX_ROLE_EDGE, "bad segment role");
    TGX_REQUIRE(m->seg_width[s] > 0 && m->seg_stride[s] >= m->seg_width[s], "bad segment %d", s);
    Role& r = *roles[role];
    if (r.n == kRoleSegs) return unsupported("two fields of a role");
    r.f[r.n++] = Field{m->seg_dev[s], nullptr, m->seg_stride[s], m->seg_width[s], r.width, k};
    v.in[s] = r.f[r.n - 1];
    v.in_role[s] = role;
    r.width += m->seg_width[s];
    k += m->seg_width[s];
  }
  TGX_REQUIRE(k <= m->width, "inputs (%d) exceed the padded width", k);
  v.in_width = k;
  v.n_in = m->n_segments;
  if (v.dst.width == 0 || v.src.width > kSrcCols || v.dst.width > kU || v.edge.width > kEdgeCols)
    return unsupported("source fields of up to 8 floats, destination fields of 1 to 16 and edge "
                       "fields of up to 7");
  v.fold = -1;
  *out = v;
  return TGX_OK;
}

void bind_state(ProjView& v, float* state, int64_t n_dst) {
  v.pt = state;
  v.packed = v.pt + n_dst * HP;
  v.bound = v.packed + Packed::end;
}

template <typename F>
void with_act(int act, F f) {
  if (act == TGX_ACT_LEAKY_RELU) return f(std::integral_constant<int, TGX_ACT_LEAKY_RELU>{});
  if (act == TGX_ACT_RELU) return f(std::integral_constant<int, TGX_ACT_RELU>{});
  f(std::integral_constant<int, -1>{});
}

struct ProjBwdLayout {
  int edge_blocks, row_blocks;
  int64_t chunk;
  size_t dzt_off, part_off, edge_sums_off, row_sums_off, bytes;
};

// Blocks are sized for the largest occupancy (4 a CU) and 256 CUs, so the
// layout does not depend on the device.
ProjBwdLayout proj_bwd_layout(int64_t n_edges, int64_t n_dst) {
  ProjBwdLayout L{};
  int64_t c = ceil_div(n_edges, int64_t{1024});
  c = align_up(static_cast<size_t>(c < 256 ? 256 : c), 256);
  L.chunk = c;
  L.edge_blocks = static_cast<int>(ceil_div(n_edges, c));
  const int64_t rows = ceil_div(n_dst, int64_t{16});
  L.row_blocks = static_cast<int>(rows < 2048 ? rows : 2048);
  Carve carve{nullptr, 0};
  L.dzt_off = reinterpret_cast<size_t>(carve.take<float>(n_dst * HP));
  L.part_off = reinterpret_cast<size_t>(carve.take<float>(ceil_div(n_edges, int64_t{kWave}) * 2 * HP));
  L.edge_sums_off =
      reinterpret_cast<size_t>(carve.take<float>((HP * (kU + 1) + 1) * static_cast<int64_t>(L.edge_blocks)));
  L.row_sums_off =
      reinterpret_cast<size_t>(carve.take<float>(HP * kU * static_cast<int64_t>(L.row_blocks)));
  L.bytes = align_up(carve.used);
  return L;
}

}  // namespace
}  // namespace tgx

using namespace tgx;

extern "C" int tgx_edge_mlp_projected_state(int64_t n_dst, const tgx_edge_mlp* mlp,
                                            int64_t* floats) {
  TGX_REQUIRE(floats && n_dst >= 0, "bad arguments");
  ProjView v;
  const int st = proj_view(mlp, &v);
  if (st != TGX_OK) return st;
  *floats = n_dst * HP + Packed::end + n_dst;
  return TGX_OK;
}

extern "C" int tgx_edge_mlp_projected_scores(const void* col, const int32_t* dst_index,
                                             int idx_bits, int64_t n_edges, int64_t n_dst,
                                             const tgx_edge_mlp* mlp,
                                             const float* w1, const float* b1, const float* w2,
                                             const float* b2, float* state, float* scores,
                                             void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n_edges >= 0 && n_dst >= 0, "bad sizes");
  ProjView v;
  const int st = proj_view(mlp, &v);
  if (st != TGX_OK) return st;
  if (n_edges == 0) return TGX_OK;
  TGX_REQUIRE(col && dst_index && state && scores && w1 && w2, "null pointer");
  for (int s = 0; s < mlp->n_segments; ++s) TGX_REQUIRE(mlp->seg_dev[s], "bad segment %d", s);
  TGX_REQUIRE(reinterpret_cast<uintptr_t>(state) % 16 == 0, "state must be 16-byte aligned");
  hipStream_t hs = as_stream(stream);
  bind_state(v, state, n_dst);
  v.w1 = w1;
  v.b1 = b1;
  v.w2 = w2;
  v.b2 = b2;
  {
    TGX_PROFILE("project_nodes_kernel", hs);
    pack_weights_kernel<<<ceil_div(Packed::end, 256), 256, 0, hs>>>(v);
    TGX_LAUNCHED("pack_weights_kernel");
    project_nodes_kernel<<<ceil_div(n_dst, int64_t{256}), 256, 0, hs>>>(v, n_dst);
    TGX_LAUNCHED("project_nodes_kernel");
  }
  TGX_PROFILE("projected_scores_kernel", hs);
  with_act(v.act, [&](auto ac) {
    constexpr int ACT = decltype(ac)::value;
    const int64_t blocks = ceil_div(n_edges, int64_t{256});
    if (idx_bits == 32)
      projected_scores_kernel<int32_t, ACT><<<blocks, 256, 0, hs>>>(
          static_cast<const int32_t*>(col), dst_index, n_edges, v, scores);
    else
      projected_scores_kernel<int64_t, ACT><<<blocks, 256, 0, hs>>>(
          static_cast<const int64_t*>(col), dst_index, n_edges, v, scores);
  });
  TGX_LAUNCHED("projected_scores_kernel");
  return TGX_OK;
}

extern "C" int tgx_edge_mlp_projected_workspace(int64_t n_edges, int64_t n_dst,
                                                const tgx_edge_mlp* mlp, size_t* bytes) {
  TGX_REQUIRE(bytes && n_edges >= 0 && n_dst >= 0, "bad arguments");
  ProjView v;
  const int st = proj_view(mlp, &v);
  if (st != TGX_OK) return st;
  *bytes = proj_bwd_layout(n_edges, n_dst).bytes;
  return TGX_OK;
}

extern "C" int tgx_edge_mlp_projected_backward(
    const void* row_ptr, const void* col, const int32_t* dst_index, int idx_bits, int64_t n_edges,
    int64_t n_dst, const tgx_edge_mlp* mlp, float* state, const float* lse,
    const float* out, const float* dout, const float* value, int32_t value_width,
    int fold_segment, float* dweights, float* const* dseg, void* ws, size_t ws_bytes,
    void* stream) {
  TGX_REQUIRE(idx_bits == 32 || idx_bits == 64, "idx_bits must be 32 or 64");
  TGX_REQUIRE(n_edges > 0 && n_dst > 0, "bad sizes");
  ProjView v;
  const int st = proj_view(mlp, &v);
  if (st != TGX_OK) return st;
  TGX_REQUIRE(row_ptr && col && dst_index && state && lse && out && dout && value && dweights &&
                  dseg && ws,
              "null pointer");
  TGX_REQUIRE(value_width > 0, "bad value width");
  const uintptr_t rows = reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(dout) |
                         reinterpret_cast<uintptr_t>(value) | reinterpret_cast<uintptr_t>(state);
  TGX_REQUIRE(rows % 16 == 0, "out, dout, value and state must be 16-byte aligned");
  TGX_REQUIRE(fold_segment >= -1 && fold_segment < mlp->n_segments, "bad fold segment");
  if (fold_segment >= 0)
    TGX_REQUIRE(mlp->seg_role[fold_segment] == TGX_ROLE_SRC &&
                    mlp->seg_width[fold_segment] == value_width,
                "the folded segment is a source field of the value's width");
  const ProjBwdLayout L = proj_bwd_layout(n_edges, n_dst);
  TGX_REQUIRE(ws_bytes >= L.bytes, "workspace too small: need %zu bytes", L.bytes);
  bind_state(v, state, n_dst);
  Role* const roles[3] = {&v.src, &v.dst, &v.edge};
  int at[3] = {0, 0, 0};
  for (int s = 0; s < mlp->n_segments; ++s) {
    TGX_REQUIRE(mlp->seg_dev[s] && dseg[s], "null pointer");
    const int role = mlp->seg_role[s];
    if (s == fold_segment) v.fold = at[role];
    roles[role]->f[at[role]++].grad = dseg[s];
  }
  v.lse = lse;
  v.out = out;
  v.dout = dout;
  v.value = value;
  v.value_width = value_width;
  char* const base = static_cast<char*>(ws);
  float* const dzt = reinterpret_cast<float*>(base + L.dzt_off);
  float* const part = reinterpret_cast<float*>(base + L.part_off);
  float* const edge_sums = reinterpret_cast<float*>(base + L.edge_sums_off);
  float* const row_sums = reinterpret_cast<float*>(base + L.row_sums_off);
  hipStream_t hs = as_stream(stream);
  const auto typed = [&](auto* rp, auto* cp) -> int {
    typedef std::remove_const_t<std::remove_reference_t<decltype(*rp)>> I;
    {
      TGX_PROFILE("projected_bwd_kernel", hs);
      with_act(v.act, [&](auto ac) {
        projected_bwd_kernel<I, decltype(ac)::value><<<L.edge_blocks, 256, 0, hs>>>(
            cp, dst_index, n_edges, L.chunk, v, dzt, part, edge_sums);
      });
      TGX_LAUNCHED("projected_bwd_kernel");
    }
    TGX_PROFILE("projected_rows_kernel", hs);
    projected_rows_kernel<I><<<L.row_blocks, 256, 0, hs>>>(rp, n_dst, v, dzt, part, row_sums);
    TGX_LAUNCHED("projected_rows_kernel");
    const int n = 2 * (v.W * v.W + v.W);
    projected_weights_kernel<<<ceil_div(n, 4), 256, 0, hs>>>(v, edge_sums, L.edge_blocks, row_sums,
                                                             L.row_blocks, dweights);
    TGX_LAUNCHED("projected_weights_kernel");
    return TGX_OK;
  };
  if (idx_bits == 32)
    return typed(static_cast<const int32_t*>(row_ptr), static_cast<const int32_t*>(col));
  return typed(static_cast<const int64_t*>(row_ptr), static_cast<const int64_t*>(col));
}

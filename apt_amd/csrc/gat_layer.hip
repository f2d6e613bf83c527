// A GAT layer over a block between its dense product and its activation, forward and backward (python/npc/model/
// gatconv.py:116-126,207-236; the arithmetic there is DGL's and torch's, an elementwise kernel or a reduction per
// step over [num_src, heads, dim] temporaries):
//   el = (ft * attn_l).sum(-1), er = (ft[:num_dst] * attn_r).sum(-1)      gat_pair_scores_*: one read of ft
//   a = edge softmax of LeakyReLU(el[src] + er[dst]), out = sum a * ft[src] + bias      the block kernels of spmm.hip
// and, from d_out,
//   dz, d_er                                       the edge kernels of spmm.hip, in slot order
//   d_ft = sum a * d_out[dst] + d_el * attn_l + d_er * attn_r, d_el = sum dz            gat_source_kernel
//   d_attn_l = sum_s d_el * ft, d_attn_r = sum_d d_er * ft, d_bias = sum_d d_out        gat_param_grad_kernel
// Everything is a stream over ft or d_out with a few registers of reduction per lane; nothing of the size of ft
// but d_ft itself is written.
// bf16: a model trained in bf16 gets what the separate operations give.  Their results are bf16 where both operands
// are, so a value that was a bf16 tensor between two of them is rounded here too (as_stored, Terms); a gradient of the
// attention vectors is what is left of large terms that cancel, and moves by several per cent with that rounding.
// Without gradients (`wide`) nothing is rounded between the rows and the result: scores, sum and result are fp32.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "feature_rows.hpp"
#include "grouped_rows.hpp"
#include "long_rows.hpp"
#include "partial_sums.hpp"

namespace apt {

int gat_block(const char* who, const int64_t* neighbors, int64_t num_dst, const int64_t* num_dst_dev, int fanout,
              const void* ft, int64_t num_src, int heads, int64_t dim, int elem_size, const float* el, const float* er,
              float slope, void* out, bool like_input, float* attn_out, const void* bias, int act, hipStream_t st);
bool gat_block_scores(const int64_t* neighbors, int64_t num_dst, int fanout, const void* ft, int64_t num_src, int heads,
                      int64_t dim, int elem_size, const void* attn_l, const void* attn_r, int attn_elem_size, float slope,
                      void* out, const void* bias, int act, hipStream_t st);
int gat_edge_grad(const char* who, const int64_t* neighbors, int64_t num_dst, int fanout, const void* ft, int64_t num_src,
                  int heads, int64_t dim, int elem_size, const float* el, const float* er, float slope, const float* attn,
                  const void* d_out, bool like_input, const int64_t* csc_indptr, float* a_edge, float* dz_edge, float* d_er,
                  hipStream_t st);

// A layer's parameters may be of another type than its rows (fp32 weights under bf16 features).
struct ParamVec {
  const void* p;
  int elem_size;
  __device__ __forceinline__ float at(int64_t i) const {
    return elem_size == 4 ? static_cast<const float*>(p)[i] : to_float<uint16_t>(static_cast<const uint16_t*>(p)[i]);
  }
  // elements i .. i + N - 1, all on their way together
  template <int N> __device__ __forceinline__ void load(int64_t i, float (&v)[N]) const {
    if (elem_size == 4) {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = static_cast<const float*>(p)[i + k];
    } else {
      uint16_t raw[N];
#pragma unroll
      for (int k = 0; k < N; ++k) raw[k] = static_cast<const uint16_t*>(p)[i + k];
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = to_float<uint16_t>(raw[k]);
    }
  }
};

// Type of what an operation of a row (T) and an attention parameter gives: bf16 only if both are.
template <typename T>
struct Terms {
  bool bf16;
  __device__ __forceinline__ explicit Terms(const ParamVec& attn, int wide = 0)
      : bf16(sizeof(T) == 2 && attn.elem_size == 2 && !wide) {}
  __device__ __forceinline__ float operator()(float v) const { return bf16 ? as_stored<uint16_t>(v) : v; }
};

// el and er of a row by LPH lanes per head (VEC features each), heads * LPH lanes per row padded to LPR: the lanes of
// a head reduce with xor shuffles.
template <typename T, int VEC, int LPH, int LPR>
__global__ __launch_bounds__(kAggBlock) void gat_pair_scores_kernel(const T* __restrict__ x, int64_t num_rows,
                                                                    int64_t num_dst, int heads, ParamVec attn_l,
                                                                    ParamVec attn_r, int wide, float* __restrict__ el,
                                                                    float* __restrict__ er) {
  constexpr int kGroups = kAggBlock / LPR;
  constexpr int kRows = 4;
  const int grp = threadIdx.x / LPR, l = threadIdx.x % LPR;
  const bool live = l < heads * LPH;
  const int h = live ? l / LPH : 0;
  const int64_t row_len = static_cast<int64_t>(heads) * VEC * LPH;
  float al[VEC], ar[VEC];
  attn_l.load(live ? l * VEC : 0, al);
  attn_r.load(live ? l * VEC : 0, ar);
  const Terms<T> term(attn_l, wide);
  const int64_t step = static_cast<int64_t>(gridDim.x) * kGroups;
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * kGroups + grp; r0 < num_rows; r0 += kRows * step) {
    Row<T, VEC> v[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q)
      v[q] = load_row<T, VEC>(x, min(r0 + q * step, num_rows - 1) * row_len + (live ? l * VEC : 0));
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const int64_t r = r0 + q * step;
      if (r >= num_rows) break;   // group-uniform
      float sl = 0.f, sr = 0.f;
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const float f = live ? row_elem<T, VEC>(v[q], k) : 0.f;
        sl += term(f * al[k]);
        sr += term(f * ar[k]);
      }
#pragma unroll
      for (int off = LPH / 2; off > 0; off >>= 1) {
        sl += __shfl_xor(sl, off, kWave);
        sr += __shfl_xor(sr, off, kWave);
      }
      if (live && l % LPH == 0) {
        el[r * heads + h] = term(sl);
        if (r < num_dst) er[r * heads + h] = term(sr);
      }
    }
  }
}

// Any heads and dim: a wavefront per (row, head).
template <typename T>
__global__ __launch_bounds__(kAggBlock) void gat_pair_scores_any_kernel(const T* __restrict__ x, int64_t num_rows,
                                                                        int64_t num_dst, int heads, int64_t dim,
                                                                        ParamVec attn_l, ParamVec attn_r, int wide,
                                                                        float* __restrict__ el, float* __restrict__ er) {
  const int lane = threadIdx.x % kWave;
  const Terms<T> term(attn_l, wide);
  const int64_t items = num_rows * heads;
  for (int64_t it = static_cast<int64_t>(blockIdx.x) * kAggWaves + threadIdx.x / kWave; it < items;
       it += static_cast<int64_t>(gridDim.x) * kAggWaves) {
    const int h = static_cast<int>(it % heads);
    float sl = 0.f, sr = 0.f;
    for (int64_t d = lane; d < dim; d += kWave) {
      const float v = to_float<T>(x[it * dim + d]);
      sl += term(v * attn_l.at(h * dim + d));
      sr += term(v * attn_r.at(h * dim + d));
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      sl += __shfl_down(sl, off, kWave);
      sr += __shfl_down(sr, off, kWave);
    }
    if (lane == 0) {
      el[it] = term(sl);
      if (it < num_dst * heads) er[it] = term(sr);
    }
  }
}

template <typename T, int VEC, int LPH>
static void launch_pair_scores_r(const void* x, int64_t n, int64_t num_dst, int heads, ParamVec al, ParamVec ar, int wide,
                                 float* el, float* er, hipStream_t st) {
#define APT_PAIR(LPR)                                                                                              \
  hipLaunchKernelGGL((gat_pair_scores_kernel<T, VEC, LPH, LPR>),                                                    \
                     dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(n, kAggBlock / LPR), 4096))),           \
                     dim3(kAggBlock), 0, st, static_cast<const T*>(x), n, num_dst, heads, al, ar, wide, el, er)
  const int lanes = heads * LPH;
  if constexpr (LPH <= 8) {
    if (lanes <= 8) {
      APT_PAIR(8);
      return;
    }
  }
  if constexpr (LPH <= 16) {
    if (lanes <= 16) {
      APT_PAIR(16);
      return;
    }
  }
  if constexpr (LPH <= 32) {
    if (lanes <= 32) {
      APT_PAIR(32);
      return;
    }
  }
  APT_PAIR(64);
#undef APT_PAIR
}

template <typename T, int VEC>
static bool launch_pair_scores(const void* x, int64_t n, int64_t num_dst, int heads, int64_t dim, ParamVec al, ParamVec ar,
                               int wide, float* el, float* er, hipStream_t st) {
  const int64_t lph = dim / VEC;
  if (dim % VEC != 0 || (lph & (lph - 1)) != 0 || heads * lph > kWave || (reinterpret_cast<uintptr_t>(x) & 15) != 0)
    return false;
  switch (lph) {
    case 1: launch_pair_scores_r<T, VEC, 1>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    case 2: launch_pair_scores_r<T, VEC, 2>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    case 4: launch_pair_scores_r<T, VEC, 4>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    case 8: launch_pair_scores_r<T, VEC, 8>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    case 16: launch_pair_scores_r<T, VEC, 16>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    case 32: launch_pair_scores_r<T, VEC, 32>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
    default: launch_pair_scores_r<T, VEC, 64>(x, n, num_dst, heads, al, ar, wide, el, er, st); return true;
  }
}

// ------------------------------------------------------------------ backward, source half
// As source_sum_kernel (block_grad.hip): a lane group per source row, hubs shared by the workgroup, rows too long for one
// workgroup cut into chunks (long_rows.hpp; a chunk's sum: the row's features, then the heads' logit gradients).
constexpr int kGatHubEdges = 16;
constexpr int kGatHubList = 1024;
constexpr int kGatSourceBlocks = 2048;      // twice as many where a lane reads single elements

struct GatSourceParams {
  const void* indptr;       // offsets of the sources in `index`
  const void* index;        // per edge: its slot (uint32_t), or its destination (int64_t) with its edge id in `eids`
  const int64_t* eids;
  uint32_t fanout;
  const float* attn;        // attention weight and logit gradient, [slot or edge id, heads]
  const float* dz;
  const void* d_out;        // [num_dst, heads * dim]
  const float* d_er;        // [num_dst, heads]
  ParamVec attn_l, attn_r;  // [heads, dim]
  int64_t num_dst, num_src;
  int heads;
  int64_t dim;              // per head
  void* d_ft;               // [num_src, heads * dim]
  float* d_el;              // [num_src, heads]
  LongRows lng;
};

// VEC consecutive features of a row belong to at most two heads (dim >= VEC): h0, and h1 from element `cut` on.
// Nearly all sources have one or two edges, so a row is a chain of three dependent reads (offsets, edges, rows of the
// destinations) and little else: a group has kRows rows in flight with their first edges, loads stand outside branches
// (a conversion inside one waits for its load), and what depends on the columns alone (heads, parameters) is taken out
// of the loop over the rows.  Rows and hubs are dealt as in block_grad.hip (grouped_rows.hpp).  124 k rows of 4 x 64 bf16,
// 261 k edges (63 MB written, 134 MB of destinations' rows read): 65 us, 61 when four neighbouring rows were a workgroup's
// (grouped_rows.hpp says why they are not); 72 with four rows in flight (161 registers instead of 111), neighbouring rows on
// different XCDs and every hub a workgroup's; 193 with a wavefront per row, loads in branches and the heads worked out per
// row.  (Three or four rows in flight where a lane reads one element: no faster.)
// Workgroups, 2048 / 4096, whole backward pass of 240 k sources 500 k edges, us: 2 x 101 fp32 812 / 759, 4 x 64 fp32 361 / 369,
// bf16 238 / 240; 124 k sampled rows of 4 x 64 bf16, the kernel alone, 41 / 43.
// TWO: a lane's features may belong to two heads.
template <typename T, int VEC, int LPR, typename I, bool TWO>
__global__ __launch_bounds__(kAggBlock) void gat_source_kernel(GatSourceParams p) {
  constexpr int kGroups = kAggBlock / LPR;
  constexpr int kRows = 2;     // rows of a group in flight,
  constexpr int kHead = 2;     // with their first edges
  constexpr int kChunk = LPR < 32 ? LPR : 32;   // edges of a hub that are looked up at once
  constexpr int kUnroll = 4;
  __shared__ int s_hub[kGatHubList];   // short hubs from the front, longer ones from the back
  __shared__ int s_hubs[2];
  __shared__ float s_sum[kGroups][LPR * (VEC + 2)];
  __shared__ uint32_t s_wave[kAggWaves], s_where[2];
  const int grp = threadIdx.x / LPR, l = threadIdx.x % LPR;
  const I* indptr = static_cast<const I*>(p.indptr);
  const I* index = static_cast<const I*>(p.index);
  const T* d_out = static_cast<const T*>(p.d_out);
  T* d_ft = static_cast<T*>(p.d_ft);
  const int64_t row_len = p.heads * p.dim;
  const Terms<T> term(p.attn_l);
  if (threadIdx.x == 0) s_hubs[0] = s_hubs[1] = 0;
  __syncthreads();
  struct Cols {
    int64_t c;
    int h0, h1, cut;
    bool live, start;   // start: the lane's first feature is its head's
    float al[VEC], ar[VEC];
  };
  auto columns = [&](int64_t c0) {
    Cols k;
    k.c = c0 + static_cast<int64_t>(l) * VEC;
    k.live = k.c < row_len;
    k.h0 = k.live ? static_cast<int>(k.c / p.dim) : 0;
    k.start = k.c == k.h0 * p.dim;
    k.cut = static_cast<int>(min(static_cast<int64_t>(VEC), (k.h0 + 1) * p.dim - k.c));
    k.h1 = k.cut < VEC ? k.h0 + 1 : k.h0;
    p.attn_l.load(k.live ? k.c : 0, k.al);
    p.attn_r.load(k.live ? k.c : 0, k.ar);
    return k;
  };
  struct Acc {
    float v[VEC];
    float el0, el1;
  };
  auto clear = [](Acc& a) {
#pragma unroll
    for (int k = 0; k < VEC; ++k) a.v[k] = 0.f;
    a.el0 = a.el1 = 0.f;
  };
  // lane j of the group holds edge j: its destination (-1: none) and where its weights are
  auto edge_of = [&](int64_t at, int64_t end, int64_t& dst, int64_t& weight) {
    const bool mine = at < end;
    const I v = index[mine ? at : 0];
    if constexpr (sizeof(I) == 4) {
      weight = static_cast<int64_t>(v);
      dst = static_cast<int64_t>(v / p.fanout);
    } else {
      weight = p.eids[mine ? at : 0];
      dst = static_cast<int64_t>(v);
    }
    if (!mine || dst >= p.num_dst) dst = -1;
  };
  // Edges that the group's lanes hold (none beyond n), all on their way before the first is used.
  struct Loaded {
    Row<T, VEC> v[kUnroll];
    float a0[kUnroll], z0[kUnroll], a1[kUnroll], z1[kUnroll];
    bool ok[kUnroll];
  };
  auto load_edges = [&](int64_t my_dst, int64_t my_weight, int e0, int n, const Cols& col, int count, Loaded& o) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (u >= count) break;
      // in the place of a missing edge, the last one again: its lines are on their way already
      const int j = max(min(min(e0 + u, n - 1), LPR - 1), 0);
      const int64_t d = __shfl(my_dst, j, LPR), w = __shfl(my_weight, j, LPR);
      o.ok[u] = e0 + u < n && d >= 0;
      const int64_t at = d >= 0 ? w * p.heads : 0;
      o.v[u] = load_row<T, VEC>(d_out, (d >= 0 ? d * row_len : 0) + (col.live ? col.c : 0));
      o.a0[u] = p.attn[at + col.h0];
      o.z0[u] = p.dz[at + col.h0];
      if (TWO) {
        o.a1[u] = p.attn[at + (col.live ? col.h1 : 0)];
        o.z1[u] = p.dz[at + (col.live ? col.h1 : 0)];
      }
    }
  };
  auto sum_edges = [&](const Loaded& o, const Cols& col, int count, Acc& acc) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (u >= count) break;
      if (!o.ok[u]) continue;
#pragma unroll
      for (int k = 0; k < VEC; ++k) acc.v[k] += (!TWO || k < col.cut ? o.a0[u] : o.a1[u]) * row_elem<T, VEC>(o.v[u], k);
      acc.el0 += o.z0[u];
      if (TWO) acc.el1 += o.z1[u];
    }
  };
  auto add_edges = [&](int64_t my_dst, int64_t my_weight, int from, int n, const Cols& col, Acc& acc) {
    for (int e0 = from; e0 < n; e0 += kUnroll) {
      Loaded o;
      load_edges(my_dst, my_weight, e0, n, col, kUnroll, o);
      sum_edges(o, col, kUnroll, acc);
    }
  };
  auto finish = [&](int64_t r, const Cols& col, const Acc& acc) {
    if (!col.live) return;
    const float e0 = term(acc.el0), e1 = term(acc.el1);
    float r0 = 0.f, r1 = 0.f;
    if (r < p.num_dst) {
      r0 = term(p.d_er[r * p.heads + col.h0]);
      if (TWO) r1 = term(p.d_er[r * p.heads + col.h1]);
    }
    float out[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const bool first = !TWO || k < col.cut;
      out[k] = as_stored<T>(acc.v[k]);
      if (r < p.num_dst) out[k] = as_stored<T>(out[k] + as_stored<T>((first ? r0 : r1) * col.ar[k]));
      out[k] += as_stored<T>((first ? e0 : e1) * col.al[k]);
    }
    if (col.start) p.d_el[r * p.heads + col.h0] = e0;
    if (TWO && col.cut < VEC) p.d_el[r * p.heads + col.h1] = e1;
    store_vec<T, VEC>(d_ft, r * row_len + col.c, out);
  };
  // acc += the edges [lo, hi), every kGroups-th by this group
  auto add_span = [&](int64_t lo, int64_t hi, const Cols& col, Acc& acc) {
    for (int64_t e = lo + grp; e < hi; e += kAggBlock) {
      int64_t d, w;
      edge_of(e + l * kGroups, hi, d, w);
      add_edges(d, w, 0, static_cast<int>(min((hi - e + kGroups - 1) / kGroups, static_cast<int64_t>(LPR))), col, acc);
    }
  };
  // The groups' sums together, in order, for the first group.
  auto over_groups = [&](Acc& acc) {
#pragma unroll
    for (int k = 0; k < VEC; ++k) s_sum[grp][k * LPR + l] = acc.v[k];
    s_sum[grp][VEC * LPR + l] = acc.el0;
    s_sum[grp][(VEC + 1) * LPR + l] = acc.el1;
    __syncthreads();
    if (grp == 0) {
      clear(acc);
#pragma unroll 1
      for (int g = 0; g < kGroups; ++g) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc.v[k] += s_sum[g][k * LPR + l];
        acc.el0 += s_sum[g][VEC * LPR + l];
        acc.el1 += s_sum[g][(VEC + 1) * LPR + l];
      }
    }
    __syncthreads();
  };
  const int64_t row_groups = static_cast<int64_t>(gridDim.x) * kGroups;
  for (int64_t c0 = 0; c0 < row_len; c0 += LPR * VEC) {
    const Cols col = columns(c0);
    for (int64_t r0 = group_row<kGroups>(grp, gridDim.x); r0 < p.num_src; r0 += kRows * row_groups) {
      int64_t lo[kRows], hi[kRows], dst[kRows], weight[kRows];
      int n[kRows];     // edges; a hub's are left for later
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        const int64_t r = r0 + q * row_groups;
        const I a = indptr[min(r, p.num_src - 1)], b = indptr[min(r, p.num_src - 1) + 1];
        lo[q] = static_cast<int64_t>(a);
        hi[q] = lo[q] + static_cast<int64_t>(b - a) * (r < p.num_src);   // (a condition would wait for the load)
      }
#pragma unroll
      for (int q = 0; q < kRows; ++q) edge_of(lo[q] + l, hi[q], dst[q], weight[q]);
      Loaded head[kRows];
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        n[q] = hi[q] - lo[q] > kGatHubEdges ? 0 : static_cast<int>(hi[q] - lo[q]);
        load_edges(dst[q], weight[q], 0, n[q], col, kHead, head[q]);
      }
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        const int64_t r = r0 + q * row_groups;
        if (r >= p.num_src) break;
        if (hi[q] - lo[q] > kGatHubEdges) {
          if (l == 0 && c0 == 0 && (p.lng.slots == 0 || hi[q] - lo[q] <= p.lng.longer)) {
            if (hi[q] - lo[q] <= hub_shared<LPR>()) s_hub[atomicAdd(&s_hubs[0], 1)] = static_cast<int>(r);
            else s_hub[kGatHubList - 1 - atomicAdd(&s_hubs[1], 1)] = static_cast<int>(r);
          }
          continue;
        }
        Acc acc;
        clear(acc);
        sum_edges(head[q], col, kHead, acc);
        add_edges(dst[q], weight[q], kHead, min(n[q], LPR), col, acc);
        for (int e = LPR; e < n[q]; e += LPR) {   // LPR < kGatHubEdges only
          int64_t d, w;
          edge_of(lo[q] + e + l, hi[q], d, w);
          add_edges(d, w, 0, min(n[q] - e, LPR), col, acc);
        }
        finish(r, col, acc);
      }
    }
  }
  __syncthreads();
  const bool apiece = s_hubs[0] >= hubs_apiece<kGroups>();
  const int hubs = apiece ? s_hubs[0] : 0, shared = s_hubs[1] + (apiece ? 0 : s_hubs[0]);
  for (int i = grp; i < hubs; i += kGroups) {
    const int64_t r = s_hub[i];
    const int64_t lo = static_cast<int64_t>(indptr[r]), hi = static_cast<int64_t>(indptr[r + 1]);
    for (int64_t c0 = 0; c0 < row_len; c0 += LPR * VEC) {
      const Cols col = columns(c0);
      Acc acc;
      clear(acc);
      for (int64_t e = lo; e < hi; e += kChunk) {
        int64_t d, w;
        edge_of(l < kChunk ? e + l : hi, hi, d, w);
        const int n = static_cast<int>(min(hi - e, static_cast<int64_t>(kChunk)));
#pragma unroll 1
        for (int f = 0; f < n; f += kGatHubEdges) {   // one rounding of the long sum for each of these
          Acc run;
          clear(run);
          add_edges(d, w, f, min(n, f + kGatHubEdges), col, run);
#pragma unroll
          for (int k = 0; k < VEC; ++k) acc.v[k] += run.v[k];
          acc.el0 += run.el0;
          acc.el1 += run.el1;
        }
      }
      finish(r, col, acc);
    }
  }
  for (int i = 0; i < shared; ++i) {
    const int64_t r = i < s_hubs[1] ? s_hub[kGatHubList - 1 - i] : s_hub[i - s_hubs[1]];
    const int64_t lo = static_cast<int64_t>(indptr[r]), hi = static_cast<int64_t>(indptr[r + 1]);
    for (int64_t c0 = 0; c0 < row_len; c0 += LPR * VEC) {
      const Cols col = columns(c0);
      Acc acc;
      clear(acc);
      add_span(lo, hi, col, acc);   // (all groups have some of the edges)
      over_groups(acc);
      if (grp == 0) finish(r, col, acc);
    }
  }
  if (p.lng.slots == 0) return;
  LongChunks<kAggBlock, I> chunks(p.lng, indptr);
  chunks.number(s_wave);
  const int64_t width = row_len + p.heads;
  for (uint32_t q = blockIdx.x; q < chunks.all; q += gridDim.x) {   // block-uniform
    const auto chunk = chunks.find(q, s_where);
    float* sum = p.lng.part + static_cast<int64_t>(q) * width;
    for (int64_t c0 = 0; c0 < row_len; c0 += LPR * VEC) {
      const Cols col = columns(c0);
      Acc acc;
      clear(acc);
      add_span(chunk.from, chunk.to, col, acc);
      over_groups(acc);
      if (grp == 0 && col.live) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) sum[col.c + k] = acc.v[k];
        if (col.start) sum[row_len + col.h0] = acc.el0;
        if (TWO && col.cut < VEC) sum[row_len + col.h1] = acc.el1;
      }
    }
    if (!chunks.last_of_row(chunk, s_where)) continue;
    const float* part = p.lng.part + static_cast<int64_t>(q - chunk.index) * width;
    for (int64_t c0 = 0; c0 < row_len; c0 += LPR * VEC) {
      const Cols col = columns(c0);
      Acc acc;
      clear(acc);
      for (uint32_t g = grp; g < chunk.count && col.live; g += kGroups) {
        const float* at = part + static_cast<int64_t>(g) * width;
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc.v[k] += at[col.c + k];
        acc.el0 += at[row_len + col.h0];
        if (TWO) acc.el1 += at[row_len + col.h1];
      }
      over_groups(acc);
      if (grp == 0) finish(chunk.row, col, acc);
    }
  }
}

template <typename T, int VEC, typename I, bool TWO>
static void launch_gat_source_as(const GatSourceParams& p, int64_t num_edges, hipStream_t st) {
  const int64_t per_row = ceil_div(p.heads * p.dim, VEC);
#define APT_GAT_SOURCE(LPR)                                                                                        \
  do {                                                                                                            \
    const int64_t for_edges = std::max(std::min(p.num_src, num_edges / (kAggBlock / LPR * kGatHubEdges)),         \
                                       p.lng.slots > 0 ? long_chunks(num_edges) : 0);                             \
    const int64_t blocks = even_grid(std::max(ceil_div(p.num_src, kGatHubList),                                   \
                                              std::min<int64_t>(std::max(ceil_div(p.num_src, 4 * kAggBlock / LPR), for_edges), \
                                                                kGatSourceBlocks * (VEC == 1 ? 2 : 1))));         \
    hipLaunchKernelGGL((gat_source_kernel<T, VEC, LPR, I, TWO>), dim3(static_cast<unsigned>(blocks)), dim3(kAggBlock), 0, st, p); \
  } while (0)
  if (per_row <= 8) APT_GAT_SOURCE(8);
  else if (per_row <= 16) APT_GAT_SOURCE(16);
  else if (per_row <= 32) APT_GAT_SOURCE(32);
  else APT_GAT_SOURCE(64);
#undef APT_GAT_SOURCE
}

template <typename T, int VEC, typename I>
static void launch_gat_source(const GatSourceParams& p, int64_t num_edges, hipStream_t st) {
  if (VEC > 1 && p.dim % VEC != 0) launch_gat_source_as<T, VEC, I, (VEC > 1)>(p, num_edges, st);
  else launch_gat_source_as<T, VEC, I, false>(p, num_edges, st);
}

template <typename T, typename I>
static void launch_gat_source_t(const GatSourceParams& p, int64_t num_edges, hipStream_t st) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(p.d_out) | reinterpret_cast<uintptr_t>(p.d_ft)) & 15) == 0;
  if constexpr (sizeof(T) == 2) {   // 16 bytes a lane: twice the rows in a wavefront
    if (aligned && (p.heads * p.dim) % 8 == 0 && p.dim >= 8) {
      launch_gat_source<T, 8, I>(p, num_edges, st);
      return;
    }
  }
  if (aligned && (p.heads * p.dim) % 4 == 0 && p.dim >= 4) launch_gat_source<T, 4, I>(p, num_edges, st);
  else launch_gat_source<T, 1, I>(p, num_edges, st);
}

// ------------------------------------------------------------------ backward, parameters
// Column sums over the rows: a thread has VEC columns of every so many-th row, first of those that are destinations too,
// then of the others, which have nothing but ft.  Bound by reading ft and d_out once; kUnroll rows of a lane group are on
// their way (loads outside branches: a conversion inside one waits for its load).  124 k rows of 4 x 64 bf16, 19 k of
// them destinations: 22 us (73 MB), 33 with the loads in branches and the rows in one
// piece per workgroup.
// TwoHeads: a lane's features may belong to two heads.
constexpr int kParamBlocks = 1024;       // at the most

template <typename T> struct TwoHeads {};
template <typename T> struct ParamRow {
  using Elem = T;
  static constexpr bool kTwo = false;
};
template <typename T> struct ParamRow<TwoHeads<T>> {
  using Elem = T;
  static constexpr bool kTwo = true;
};

template <typename R, int VEC>
__global__ __launch_bounds__(kAggBlock) void gat_param_grad_kernel(const typename ParamRow<R>::Elem* __restrict__ ft,
                                                                   const typename ParamRow<R>::Elem* __restrict__ d_out,
                                                                   const float* __restrict__ d_el,
                                                                   const float* __restrict__ d_er, int64_t num_src,
                                                                   int64_t num_dst, int heads, int64_t dim, int lanes,
                                                                   float* __restrict__ part, ParamVec attn_l) {
  using T = typename ParamRow<R>::Elem;
  constexpr bool TWO = ParamRow<R>::kTwo;
  constexpr int kUnroll = 8;
  const Terms<T> term(attn_l);
  __shared__ float s_sum[3 * VEC][kAggBlock];
  const int64_t row_len = heads * dim;
  const int groups = kAggBlock / lanes, grp = threadIdx.x / lanes, l = threadIdx.x % lanes;
  const int64_t first = static_cast<int64_t>(grp) * gridDim.x + blockIdx.x, step = static_cast<int64_t>(groups) * gridDim.x;
  float* out = part + static_cast<int64_t>(blockIdx.x) * 3 * row_len;
  for (int64_t c0 = 0; c0 < row_len; c0 += static_cast<int64_t>(lanes) * VEC) {
    const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
    const bool live = c < row_len;
    const int64_t at = live ? c : 0;
    const int h0 = static_cast<int>(at / dim);
    const int cut = static_cast<int>(min(static_cast<int64_t>(VEC), (h0 + 1) * dim - at));
    const int h1 = cut < VEC ? h0 + 1 : h0;
    float sl[VEC], sr[VEC], sb[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) sl[k] = sr[k] = sb[k] = 0.f;
    auto rows = [&](int64_t from, int64_t to, auto both) {
      for (int64_t r0 = from + first; r0 < to; r0 += kUnroll * step) {
        Row<T, VEC> v[kUnroll], o[kUnroll];
        float l0[kUnroll], l1[kUnroll], e0[kUnroll], e1[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const int64_t r = min(r0 + u * step, to - 1);
          v[u] = load_row<T, VEC>(ft, r * row_len + at);
          l0[u] = d_el[r * heads + h0];
          if (TWO) l1[u] = d_el[r * heads + h1];
          if constexpr (decltype(both)::value) {
            o[u] = load_row<T, VEC>(d_out, r * row_len + at);
            e0[u] = d_er[r * heads + h0];
            if (TWO) e1[u] = d_er[r * heads + h1];
          }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          if (r0 + u * step >= to) break;   // group-uniform
          if constexpr (decltype(both)::value) {
            e0[u] = term(e0[u]);
            if (TWO) e1[u] = term(e1[u]);
          }
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            const bool own = !TWO || k < cut;
            const float f = row_elem<T, VEC>(v[u], k);
            sl[k] += term((own ? l0[u] : l1[u]) * f);
            if constexpr (decltype(both)::value) {
              sr[k] += term((own ? e0[u] : e1[u]) * f);
              sb[k] += row_elem<T, VEC>(o[u], k);
            }
          }
        }
      }
    };
    // Single elements: nothing that is added stands in a branch, since the loads would move into it, each waited for there
    // (500 k rows of 2 x 101 fp32 264 us instead of 113; rows of vectors are the faster with the branch, 4 x 64 fp32 118 and
    // 142).  `some`: of a turn's rows some are missing; the first is read in their place and counts as zeros.
    auto singles = [&](int64_t from, int64_t to, auto both) {
      auto turn = [&](int64_t r0, auto some) {
        T v[kUnroll], o[kUnroll];
        float l0[kUnroll], e0[kUnroll];
        bool in[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          in[u] = !decltype(some)::value || r0 + u * step < to;
          const int64_t r = in[u] ? r0 + u * step : r0;
          v[u] = ft[r * row_len + at];
          l0[u] = d_el[r * heads + h0];
          if constexpr (decltype(both)::value) {
            o[u] = d_out[r * row_len + at];
            e0[u] = d_er[r * heads + h0];
          }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const float f = to_float<T>(v[u]);
          sl[0] += in[u] ? term(l0[u] * f) : 0.f;
          if constexpr (decltype(both)::value) {
            sr[0] += in[u] ? term(term(e0[u]) * f) : 0.f;
            sb[0] += in[u] ? to_float<T>(o[u]) : 0.f;
          }
        }
      };
      int64_t r0 = from + first;
      for (; r0 + (kUnroll - 1) * step < to; r0 += kUnroll * step) turn(r0, std::false_type{});
      for (; r0 < to; r0 += kUnroll * step) turn(r0, std::true_type{});
    };
    if constexpr (VEC == 1) {
      singles(0, num_dst, std::true_type{});
      singles(num_dst, num_src, std::false_type{});
    } else {
      rows(0, num_dst, std::true_type{});
      rows(num_dst, num_src, std::false_type{});
    }
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      s_sum[k][threadIdx.x] = sl[k];
      s_sum[VEC + k][threadIdx.x] = sr[k];
      s_sum[2 * VEC + k][threadIdx.x] = sb[k];
    }
    __syncthreads();
    if (grp == 0 && live) {
#pragma unroll
      for (int k = 0; k < VEC; ++k)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          float sum = 0.f;
          for (int g = 0; g < groups; ++g) sum += s_sum[q * VEC + k][g * lanes + l];
          out[q * row_len + c + k] = sum;
        }
    }
    __syncthreads();
  }
}

static int64_t param_blocks(int64_t num_src) { return std::min<int64_t>(std::max<int64_t>(ceil_div(num_src, 16), 1), kParamBlocks); }

// -> the number of partial sums that it leaves.  Half as many workgroups where a lane reads eight elements: 122 k rows of
// 4 x 64 bf16, whole backward pass, 149 us (158 with 1024, 164 with 2048); of 2 x 101 fp32, one by one, 389 / 354 / 360.
template <typename T>
static int launch_param_grad(const void* ft, const void* d_out, const float* d_el, const float* d_er, int64_t num_src,
                             int64_t num_dst, int heads, int64_t dim, float* part, ParamVec attn_l, hipStream_t st) {
  const int64_t row_len = heads * dim;
  const bool aligned = ((reinterpret_cast<uintptr_t>(ft) | reinterpret_cast<uintptr_t>(d_out)) & 15) == 0;
  constexpr int kWide = 16 / sizeof(T);
  const int vec = aligned && row_len % kWide == 0 && dim >= kWide ? kWide : aligned && row_len % 4 == 0 && dim >= 4 ? 4 : 1;
  int lanes = 8;
  while (lanes < kAggBlock && lanes * vec < row_len) lanes <<= 1;
  const int64_t blocks = std::min<int64_t>(param_blocks(num_src), vec == 8 ? kParamBlocks / 2 : kParamBlocks);
  const dim3 grid(static_cast<unsigned>(blocks)), block(kAggBlock);
#define APT_PARAM(R, V)                                                                                            \
  hipLaunchKernelGGL((gat_param_grad_kernel<R, V>), grid, block, 0, st, static_cast<const T*>(ft),                  \
                     static_cast<const T*>(d_out), d_el, d_er, num_src, num_dst, heads, dim, lanes, part, attn_l)
  if (vec == kWide) {
    if (dim % kWide == 0) APT_PARAM(T, kWide);
    else APT_PARAM(TwoHeads<T>, kWide);
  } else if (vec == 4) {
    if (dim % 4 == 0) APT_PARAM(T, 4);
    else APT_PARAM(TwoHeads<T>, 4);
  } else {
    APT_PARAM(T, 1);
  }
#undef APT_PARAM
  return static_cast<int>(blocks);
}

// d_attn_l, d_attn_r (of one type) and d_bias (of the rows') from `splits` partials of 3 * n; zeros from none.
static int gat_param_sums(const float* part, int splits, int64_t n, int elem_size, int attn_elem_size, void* d_attn_l,
                          void* d_attn_r, void* d_bias, hipStream_t st) {
  if (d_attn_l == nullptr && d_attn_r == nullptr && d_bias == nullptr) return APT_OK;
  if (attn_elem_size == elem_size) {
    if (elem_size == 4) launch_partial_sums<float, float>(part, 3 * n, splits, d_attn_l, n, d_attn_r, n, d_bias, n, st);
    else launch_partial_sums<uint16_t, uint16_t>(part, 3 * n, splits, d_attn_l, n, d_attn_r, n, d_bias, n, st);
    APT_LAUNCH_CHECK("partial_sums_kernel");
    return APT_OK;
  }
  if (attn_elem_size == 4) launch_partial_sums<float, float>(part, 3 * n, splits, d_attn_l, n, d_attn_r, n, nullptr, 0, st);
  else launch_partial_sums<uint16_t, uint16_t>(part, 3 * n, splits, d_attn_l, n, d_attn_r, n, nullptr, 0, st);
  APT_LAUNCH_CHECK("partial_sums_kernel");
  if (d_bias == nullptr) return APT_OK;
  if (elem_size == 4) launch_partial_sums<float, float>(part + 2 * n, 3 * n, splits, d_bias, n, nullptr, 0, nullptr, 0, st);
  else launch_partial_sums<uint16_t, uint16_t>(part + 2 * n, 3 * n, splits, d_bias, n, nullptr, 0, nullptr, 0, st);
  APT_LAUNCH_CHECK("partial_sums_kernel");
  return APT_OK;
}

static size_t align256(size_t x) { return (x + 255) / 256 * 256; }

}  // namespace apt

extern "C" int apt_gat_layer(const int64_t* neighbors, int64_t num_dst, int fanout, const void* ft, int64_t num_src,
                             int heads, int64_t dim, int elem_size, const void* attn_l, const void* attn_r,
                             int attn_elem_size, const void* bias, int relu, float negative_slope, int wide, float* el,
                             float* er, void* out, float* attn_out, void* stream) {
  using namespace apt;
  const char* who = "apt_gat_layer";
  APT_REQUIRE(num_dst >= 0 && num_dst <= num_src && fanout > 0 && heads > 0 && dim > 0, APT_EINVAL,
              "%s: bad shape (num_dst %lld, num_src %lld, fanout %d, heads %d, dim %lld)", who, (long long)num_dst,
              (long long)num_src, fanout, heads, (long long)dim);
  APT_REQUIRE((elem_size == 2 || elem_size == 4) && (attn_elem_size == 2 || attn_elem_size == 4), APT_EINVAL,
              "%s: elem_size %d, attn_elem_size %d (4 = fp32, 2 = bf16)", who, elem_size, attn_elem_size);
  if (num_src == 0) return APT_OK;
  APT_REQUIRE(ft != nullptr && attn_l != nullptr && attn_r != nullptr && el != nullptr && (num_dst == 0 || er != nullptr),
              APT_EINVAL, "%s: a tensor is NULL", who);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const ParamVec al{attn_l, attn_elem_size}, ar{attn_r, attn_elem_size};
  const bool done = elem_size == 4 ? launch_pair_scores<float, 4>(ft, num_src, num_dst, heads, dim, al, ar, wide, el, er, st)
                                   : launch_pair_scores<uint16_t, 8>(ft, num_src, num_dst, heads, dim, al, ar, wide, el, er, st) ||
                                         launch_pair_scores<uint16_t, 4>(ft, num_src, num_dst, heads, dim, al, ar, wide, el, er, st);
  if (!done) {
    const dim3 grid(static_cast<unsigned>(std::min<int64_t>(ceil_div(num_src * heads, kAggWaves), 1 << 16))), block(kAggBlock);
    if (elem_size == 4)
      hipLaunchKernelGGL(gat_pair_scores_any_kernel<float>, grid, block, 0, st, static_cast<const float*>(ft), num_src, num_dst,
                         heads, dim, al, ar, wide, el, er);
    else
      hipLaunchKernelGGL(gat_pair_scores_any_kernel<uint16_t>, grid, block, 0, st, static_cast<const uint16_t*>(ft), num_src,
                         num_dst, heads, dim, al, ar, wide, el, er);
  }
  APT_LAUNCH_CHECK("gat_pair_scores_kernel");
  return gat_block(who, neighbors, num_dst, nullptr, fanout, ft, num_src, heads, dim, elem_size, el, er, negative_slope, out,
                   wide == 0, attn_out, bias, relu, st);
}

extern "C" int apt_gat_layer_infer(const int64_t* neighbors, int64_t num_dst, int fanout, const void* ft, int64_t num_src,
                                   int heads, int64_t dim, int elem_size, const void* attn_l, const void* attn_r,
                                   int attn_elem_size, const float* bias, int relu, float negative_slope, float* scratch,
                                   float* out, void* stream) {
  using namespace apt;
  if (num_dst > 0 && num_dst <= num_src && fanout > 0 && heads > 0 && dim > 0 && (elem_size == 2 || elem_size == 4) &&
      (attn_elem_size == 2 || attn_elem_size == 4) && neighbors != nullptr && ft != nullptr && attn_l != nullptr &&
      attn_r != nullptr && out != nullptr &&
      gat_block_scores(neighbors, num_dst, fanout, ft, num_src, heads, dim, elem_size, attn_l, attn_r, attn_elem_size,
                       negative_slope, out, bias, relu, static_cast<hipStream_t>(stream))) {
    APT_LAUNCH_CHECK("gat_ell_scores_kernel");
    return APT_OK;
  }
  return apt_gat_layer(neighbors, num_dst, fanout, ft, num_src, heads, dim, elem_size, attn_l, attn_r, attn_elem_size, bias, relu,
                       negative_slope, 1, scratch, scratch == nullptr ? nullptr : scratch + num_src * heads, out, nullptr, stream);
}

extern "C" size_t apt_gat_layer_backward_workspace_bytes(int64_t num_dst, int fanout, int64_t num_src, int heads, int64_t dim,
                                                         int64_t num_edges) {
  using namespace apt;
  if (num_dst < 0 || fanout <= 0 || num_src < 0 || heads <= 0 || dim <= 0 || num_edges < 0) return 0;
  const int64_t weights = std::max(num_dst * fanout, num_edges) * heads;
  return align256(sizeof(float) * 2 * weights) + align256(sizeof(float) * (num_dst + num_src) * heads) +
         align256(sizeof(float) * 3 * heads * dim * param_blocks(num_src)) +
         align256(sizeof(float) * long_chunks(std::max(num_dst * fanout, num_edges)) * (heads * dim + heads)) + 256;
}

extern "C" int apt_gat_layer_backward(const int64_t* neighbors, int64_t num_dst, int fanout, const void* ft,
                                      int64_t num_src, int heads, int64_t dim, int elem_size, const void* attn_l,
                                      const void* attn_r, int attn_elem_size, float negative_slope, const float* el,
                                      const float* er, const float* attn, const void* d_out, const void* indptr,
                                      const void* index, int index_bytes, const int64_t* eids, const int64_t* csc_indptr,
                                      int64_t num_edges, void* long_table, void* d_ft, void* d_attn_l, void* d_attn_r, void* d_bias,
                                      void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  const char* who = "apt_gat_layer_backward";
  APT_REQUIRE(num_dst >= 0 && num_dst <= num_src && num_src <= 0x7fffffffLL && fanout > 0 && heads > 0 && dim > 0 && num_edges >= 0,
              APT_EINVAL, "%s: bad shape (num_dst %lld, num_src %lld, fanout %d, heads %d, dim %lld)", who,
              (long long)num_dst, (long long)num_src, fanout, heads, (long long)dim);
  APT_REQUIRE((elem_size == 2 || elem_size == 4) && (attn_elem_size == 2 || attn_elem_size == 4), APT_EINVAL,
              "%s: elem_size %d, attn_elem_size %d (4 = fp32, 2 = bf16)", who, elem_size, attn_elem_size);
  APT_REQUIRE(index_bytes == 4 || (index_bytes == 8 && (eids != nullptr || num_edges == 0) && csc_indptr != nullptr), APT_EINVAL,
              "%s: index_bytes %d (4 = slots, 8 = destinations, with eids and csc_indptr)", who, index_bytes);
  APT_REQUIRE(workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
                  workspace_bytes >= apt_gat_layer_backward_workspace_bytes(num_dst, fanout, num_src, heads, dim, num_edges),
              APT_EWORKSPACE, "%s: workspace too small or not 16-byte aligned", who);
  if (num_src == 0)   // no rows: the parameters' gradients are zeros
    return gat_param_sums(static_cast<const float*>(workspace), 0, static_cast<int64_t>(heads) * dim, elem_size, attn_elem_size,
                          d_attn_l, d_attn_r, d_bias, static_cast<hipStream_t>(stream));
  APT_REQUIRE(ft != nullptr && attn_l != nullptr && attn_r != nullptr && el != nullptr && indptr != nullptr && d_ft != nullptr &&
                  (num_dst == 0 || (neighbors != nullptr && er != nullptr && attn != nullptr && d_out != nullptr &&
                                    (index != nullptr || (index_bytes == 8 && num_edges == 0)))),
              APT_EINVAL, "%s: a tensor is NULL", who);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool by_slot = index_bytes == 4;
  char* ws = static_cast<char*>(workspace);
  const int64_t weights = std::max(num_dst * fanout, num_edges) * heads;
  float* dz = reinterpret_cast<float*>(ws);
  float* a_edge = dz + weights;
  ws += align256(sizeof(float) * 2 * weights);
  float* d_er = reinterpret_cast<float*>(ws);
  float* d_el = d_er + num_dst * heads;
  ws += align256(sizeof(float) * (num_dst + num_src) * heads);
  float* part = reinterpret_cast<float*>(ws);
  ws += align256(sizeof(float) * 3 * heads * dim * param_blocks(num_src));
  if (const int rc = gat_edge_grad(who, neighbors, num_dst, fanout, ft, num_src, heads, dim, elem_size, el, er,
                                   negative_slope, attn, d_out, true, by_slot ? nullptr : csc_indptr, a_edge, dz, d_er, st))
    return rc;
  GatSourceParams p;
  p.indptr = indptr;
  p.index = index;
  p.eids = eids;
  p.fanout = static_cast<uint32_t>(fanout);
  p.attn = by_slot ? attn : a_edge;
  p.dz = dz;
  p.d_out = d_out;
  p.d_er = d_er;
  p.attn_l = ParamVec{attn_l, attn_elem_size};
  p.attn_r = ParamVec{attn_r, attn_elem_size};
  p.num_dst = num_dst;
  p.num_src = num_src;
  p.heads = heads;
  p.dim = dim;
  p.d_ft = d_ft;
  p.d_el = d_el;
  const int64_t edges = by_slot ? num_dst * fanout : num_edges;
  p.lng = long_rows(long_table, edges, reinterpret_cast<float*>(ws));
  if (num_dst == 0) {   // entry 0 of every array is read in the place of a missing edge
    p.d_out = ft;
    p.attn = p.dz = el;
  }
  if (index == nullptr || num_dst == 0) p.index = indptr;
  if (!by_slot && (eids == nullptr || num_edges == 0)) p.eids = static_cast<const int64_t*>(indptr);
  if (elem_size == 4) {
    if (by_slot) launch_gat_source_t<float, uint32_t>(p, edges, st);
    else launch_gat_source_t<float, int64_t>(p, edges, st);
  } else {
    if (by_slot) launch_gat_source_t<uint16_t, uint32_t>(p, edges, st);
    else launch_gat_source_t<uint16_t, int64_t>(p, edges, st);
  }
  APT_LAUNCH_CHECK("gat_source_kernel");
  if (d_attn_l == nullptr && d_attn_r == nullptr && d_bias == nullptr) return APT_OK;
  const int parts = elem_size == 4 ? launch_param_grad<float>(ft, d_out, d_el, d_er, num_src, num_dst, heads, dim, part, p.attn_l, st)
                                   : launch_param_grad<uint16_t>(ft, d_out, d_el, d_er, num_src, num_dst, heads, dim, part, p.attn_l, st);
  APT_LAUNCH_CHECK("gat_param_grad_kernel");
  return gat_param_sums(part, parts, static_cast<int64_t>(heads) * dim, elem_size, attn_elem_size,
                        d_attn_l, d_attn_r, d_bias, st);
}

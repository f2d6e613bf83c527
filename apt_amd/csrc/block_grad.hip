// Sums over grouped edges: dx[s, :] = sum over the edges e of s of w(e) * dz[d(e), :].  With the edges of a sampled
// block grouped by source this is the gradient of the block sum / mean towards its input; with the edges of a COO
// grouped by destination it is the COO sum (apt_coo_sum).  "Source" below is the row that is written.
//
// A lane group owns a source row, so every row is written once, in its own type, whole and in a fixed order: no
// zero-fill, no atomics, no fp32 copy of a bf16 result.  Nearly all sources of a sampled block have one or two edges;
// two rows per group are looked up at once.  Rows longer than kHubEdges are put aside: the shorter of them are added up
// by a group each afterwards, the longer by all groups of the workgroup.  Hubs have neighbouring ids (the relabel numbers
// nodes by first occurrence), so a group's rows are taken a grid apart.  Rows that are too long for one workgroup as well
// are cut into chunks (long_rows.hpp).
//
// Bound by rows of dz that come from beyond the L2 where blocks are large, hence group_row, and by chains of dependent reads
// (offsets, edges, scales, rows) where they are not, hence eight wavefronts on a SIMD (kFullSgprs).  Sum with the ordering of
// the edges, before (rows dealt to the XCDs one by one, every hub to a whole workgroup, bf16 rows converted where they were
// loaded) / now, us, fanout 15 and 10, sources drawn with density r^(1/3 - 1) and r^(1/2 - 1): 240 k sources 750 k edges
// 256 fp32 275 / 215, 256 bf16 233 / 138, 64 bf16 186 / 125, 47 bf16 264 / 175; 122 k sources 260 k edges 112 / 93, 104 / 69,
// 91 / 66, 102 / 73.  Without any skew 500 k sources 1 M edges: 307 / 290, 221 / 175, 156 / 126, 180 / 174.
#include <algorithm>

#include "common.hpp"
#include "feature_rows.hpp"
#include "grouped_rows.hpp"
#include "long_rows.hpp"

namespace apt {

constexpr int kHubEdges = 16;
constexpr int kHubList = 1024;             // rows of a workgroup at the most, so its list of hubs never overflows
constexpr int kSourceBlocks = 4096;
constexpr int kLongBlocks = 512;           // workgroups for long rows at the most

struct SourceSumParams {
  const void* indptr;      // offsets of the sources in `index`
  const void* index;       // per edge: its destination (int64_t), or its slot (uint32_t; NULL: edge e is slot e)
  uint32_t fanout;         // slots: the destination is slot / fanout ...
  const int64_t* via;      // ... or, if given, via[slot]
  const void* edata;       // slots, optional: [slots, dim] of dz's type, multiplies the destination's row
  const float* dst_scale;  // per destination, or NULL
  float scale;             // of every sum
  const void* dz;          // [num_dst, dim]
  int64_t num_dst;
  int64_t dim;
  int64_t num_src;
  void* dx;                // [num_src, dim]
  LongRows lng;
  uint32_t row_blocks;     // workgroups for the rows; those behind them take the long ones
};

// A value of lane `lane` of the group; a whole wavefront's is the same in all lanes and stands in a scalar register.
template <int LPR> __device__ __forceinline__ int group_read(int v, int lane) {
  if constexpr (LPR == kWave) return __builtin_amdgcn_readlane(v, lane);
  else return __shfl(v, lane, LPR);
}
template <int LPR> __device__ __forceinline__ uint32_t group_read(uint32_t v, int lane) {
  return static_cast<uint32_t>(group_read<LPR>(static_cast<int>(v), lane));
}
template <int LPR> __device__ __forceinline__ float group_read(float v, int lane) {
  return __int_as_float(group_read<LPR>(__float_as_int(v), lane));
}
template <int LPR> __device__ __forceinline__ int64_t group_read(int64_t v, int lane) {
  const uint32_t lo = group_read<LPR>(static_cast<uint32_t>(v), lane), hi = group_read<LPR>(static_cast<uint32_t>(v >> 32), lane);
  return static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo);
}

// I: int64_t = a block's CSR (offsets, destinations), uint32_t = apt_block_transpose (offsets, slots).
// LONG: workgroups behind those of the rows take the long rows.
template <typename T, int VEC, int LPR, typename I, bool EDATA, bool LONG>
__global__ __launch_bounds__(kAggBlock) __attribute__((amdgpu_num_sgpr(kFullSgprs))) void source_sum_kernel(SourceSumParams p) {
  constexpr int kGroups = kAggBlock / LPR;
  constexpr int kRows = 2;
  constexpr int kUnroll = 4;
  constexpr int kChunk = LPR < 32 ? LPR : 32;   // edges of a hub that are looked up at once
  __shared__ int s_hub[kHubList];
  __shared__ int s_hubs[2];
  __shared__ float s_sum[kGroups][LPR * VEC];
  __shared__ uint32_t s_wave[LONG ? kAggWaves : 1], s_where[LONG ? 2 : 1];
  const int grp = threadIdx.x / LPR, l = threadIdx.x % LPR;
  const I* indptr = static_cast<const I*>(p.indptr);
  const I* index = static_cast<const I*>(p.index);
  const T* dz = static_cast<const T*>(p.dz);
  T* dx = static_cast<T*>(p.dx);
  if (threadIdx.x == 0) s_hubs[0] = s_hubs[1] = 0;
  __syncthreads();
  struct Edge {      // lane j of a group: edge j of the row
    int64_t dst;     // -1: none
    uint32_t slot;   // EDATA only
    float scale;
  };
  // Edges at[q] of lists, where they exist (entry 0 is read in the place of others): all on their way together, step by step.
  auto look_up = [&](auto& at, const auto& mine, auto& e) {
    constexpr int kCount = sizeof(at) / sizeof(at[0]);
    I v[kCount];
    if (sizeof(I) == 8 || index != nullptr) {
#pragma unroll
      for (int q = 0; q < kCount; ++q) v[q] = index[mine[q] ? at[q] : 0];
    } else {
#pragma unroll
      for (int q = 0; q < kCount; ++q) v[q] = static_cast<I>(mine[q] ? at[q] : 0);
    }
    if (sizeof(I) == 4 && p.via != nullptr) {
#pragma unroll
      for (int q = 0; q < kCount; ++q) e[q].dst = p.via[mine[q] ? v[q] : I{0}];   // (a list without edges is not filled)
    } else {
#pragma unroll
      for (int q = 0; q < kCount; ++q) e[q].dst = sizeof(I) == 8 ? static_cast<int64_t>(v[q]) : static_cast<int64_t>(v[q] / p.fanout);
    }
#pragma unroll
    for (int q = 0; q < kCount; ++q) {
      e[q].slot = static_cast<uint32_t>(v[q]);
      if (!mine[q] || e[q].dst < 0 || e[q].dst >= p.num_dst) e[q].dst = -1;
      e[q].scale = 1.f;
    }
    if (p.dst_scale != nullptr) {
#pragma unroll
      for (int q = 0; q < kCount; ++q) e[q].scale = p.dst_scale[e[q].dst >= 0 ? e[q].dst : 0];
    }
  };
  auto edge = [&](int64_t at, bool mine) {
    const int64_t ats[1] = {at};
    const bool mines[1] = {mine};
    Edge e[1];
    look_up(ats, mines, e);
    return e[0];
  };
  const T* edata = static_cast<const T*>(p.edata);
  // acc += the rows of edges from .. n - 1 that the group's lanes hold, kUnroll on their way at once.  What is loaded in a
  // branch is converted behind all of them: a conversion inside one waits for its load.
  auto walk = [&](const Edge& my, int from, int n, int64_t c, float (&acc)[VEC]) {
    const int64_t col = min(c, p.dim - VEC);   // (lanes without columns read with the last one)
    for (int e0 = from; e0 < n; e0 += kUnroll) {
      Row<T, VEC> v[kUnroll], m[EDATA ? kUnroll : 1];
      float w[kUnroll];
      bool ok[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        ok[u] = false;
        w[u] = 0.f;
        if (e0 + u < n) {   // group-uniform
          const int64_t d = group_read<LPR>(my.dst, e0 + u);
          w[u] = group_read<LPR>(my.scale, e0 + u);
          ok[u] = d >= 0;
          v[u] = load_row<T, VEC>(dz, (d >= 0 ? d * p.dim : 0) + col);
          if constexpr (EDATA)
            m[u] = load_row<T, VEC>(edata, static_cast<int64_t>(group_read<LPR>(my.slot, e0 + u)) * p.dim + col);
        }
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        if (!ok[u]) continue;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          float f = row_elem<T, VEC>(v[u], k);
          if constexpr (EDATA) f *= row_elem<T, VEC>(m[u], k);
          acc[k] += w[u] * f;
        }
      }
    }
  };
  // acc += the edges [lo, hi), every kGroups-th by this group
  auto add_span = [&](int64_t lo, int64_t hi, int64_t c, float (&acc)[VEC]) {
    for (int64_t e = lo + grp; e < hi; e += kAggBlock) {
      const int64_t at = e + static_cast<int64_t>(l) * kGroups;
      walk(edge(at, at < hi), 0, static_cast<int>(min((hi - e + kGroups - 1) / kGroups, static_cast<int64_t>(LPR))), c, acc);
    }
  };
  // The groups' sums together, in order, for the first group.  Many groups' are read eight at a time (256 workgroups of 32 groups
  // and a hub or two each: 9 us, 17 one by one); for few groups the registers would cost more (8 bf16 a lane: 122 to 131 us).
  constexpr int kMeeting = kGroups > 8 ? 8 : 1;
  auto over_groups = [&](float (&acc)[VEC]) {
#pragma unroll
    for (int k = 0; k < VEC; ++k) s_sum[grp][l * VEC + k] = acc[k];
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        float sum = 0.f;
#pragma unroll kMeeting
        for (int g = 0; g < kGroups; ++g) sum += s_sum[g][l * VEC + k];
        acc[k] = sum;
      }
    }
    __syncthreads();
  };
  if (LONG && blockIdx.x >= p.row_blocks) {   // block-uniform
    LongChunks<kAggBlock, I> chunks(p.lng, indptr);
    chunks.number(s_wave);
    for (uint32_t q = blockIdx.x - p.row_blocks; q < chunks.all; q += gridDim.x - p.row_blocks) {
      const auto chunk = chunks.find(q, s_where);
      const float* part = p.lng.part + static_cast<int64_t>(q - chunk.index) * p.dim;   // of the row's chunks
      bool whole = false;
      for (;;) {   // the chunk's edges; then, for the workgroup that completes the row, its chunks' sums
        for (int64_t c0 = 0; c0 < p.dim; c0 += LPR * VEC) {
          const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
          const bool live = c < p.dim;
          float acc[VEC];
#pragma unroll
          for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
          if (!whole) add_span(chunk.from, chunk.to, c, acc);
          for (uint32_t g = grp; whole && g < chunk.count && live; g += kGroups)
#pragma unroll
            for (int k = 0; k < VEC; ++k) acc[k] += part[static_cast<int64_t>(g) * p.dim + c + k];
          over_groups(acc);
          if (grp == 0 && live && !whole) {
#pragma unroll
            for (int k = 0; k < VEC; ++k) p.lng.part[static_cast<int64_t>(q) * p.dim + c + k] = acc[k];
          } else if (grp == 0 && live) {
#pragma unroll
            for (int k = 0; k < VEC; ++k) acc[k] *= p.scale;
            store_vec<T, VEC>(dx, chunk.row * p.dim + c, acc);
          }
        }
        if (whole || !chunks.last_of_row(chunk, s_where)) break;
        whole = true;
      }
    }
    return;
  }
  const int64_t row_groups = static_cast<int64_t>(p.row_blocks) * kGroups;
  for (int64_t r0 = group_row<kGroups>(grp, p.row_blocks); r0 < p.num_src; r0 += kRows * row_groups) {
    int64_t lo[kRows], at[kRows];
    int n[kRows];
    bool mine[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const int64_t r = r0 + q * row_groups;
      const I a = indptr[min(r, p.num_src - 1)], b = indptr[min(r, p.num_src - 1) + 1];
      lo[q] = static_cast<int64_t>(a);
      n[q] = static_cast<int>(b - a) * (r < p.num_src);   // (a condition would wait for the load)
    }
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      at[q] = lo[q] + l;
      mine[q] = l < n[q] && n[q] <= kHubEdges;
    }
    Edge first[kRows];
    look_up(at, mine, first);
    for (int64_t c0 = 0; c0 < p.dim; c0 += LPR * VEC) {
      const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
      const bool live = c < p.dim;
#pragma unroll
      for (int q = 0; q < kRows; ++q) {
        const int64_t r = r0 + q * row_groups;
        if (r >= p.num_src || n[q] > kHubEdges) continue;   // group-uniform
        float acc[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
        walk(first[q], 0, min(n[q], LPR), c, acc);
        for (int e = LPR; e < n[q]; e += LPR)   // LPR < kHubEdges only
          walk(edge(lo[q] + e + l, e + l < n[q]), 0, min(n[q] - e, LPR), c, acc);
        if (live) {
#pragma unroll
          for (int k = 0; k < VEC; ++k) acc[k] *= p.scale;
          store_vec<T, VEC>(dx, r * p.dim + c, acc);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kRows; ++q)
      if (n[q] > kHubEdges && l == 0 && (p.lng.slots == 0 || n[q] <= static_cast<int>(p.lng.longer))) {
        if (n[q] <= hub_shared<LPR>()) s_hub[atomicAdd(&s_hubs[0], 1)] = static_cast<int>(r0 + q * row_groups);
        else s_hub[kHubList - 1 - atomicAdd(&s_hubs[1], 1)] = static_cast<int>(r0 + q * row_groups);
      }
  }
  __syncthreads();
  // (in any order: every hub is summed on its own)
  // A group each for the shorter hubs if that keeps them busy; otherwise one after the other by all groups, as the longer.
  const bool apiece = s_hubs[0] >= hubs_apiece<kGroups>();
  const int hubs = apiece ? s_hubs[0] : 0, shared = s_hubs[1] + (apiece ? 0 : s_hubs[0]);
  for (int i = grp; i < hubs; i += kGroups) {
    const int64_t r = s_hub[i];
    const int64_t lo = static_cast<int64_t>(indptr[r]);
    const int n = static_cast<int>(static_cast<int64_t>(indptr[r + 1]) - lo);
    for (int64_t c0 = 0; c0 < p.dim; c0 += LPR * VEC) {
      const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
      const bool live = c < p.dim;
      float acc[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
      for (int k0 = 0; k0 < n; k0 += kChunk) {
        const Edge my = edge(lo + k0 + l, l < kChunk && k0 + l < n);
#pragma unroll 1
        for (int e = 0; e < min(n - k0, kChunk); e += kHubEdges) {   // one rounding of the long sum for each of these
          float run[VEC];
#pragma unroll
          for (int k = 0; k < VEC; ++k) run[k] = 0.f;
          walk(my, e, min(min(n - k0, kChunk), e + kHubEdges), c, run);
#pragma unroll
          for (int k = 0; k < VEC; ++k) acc[k] += run[k];
        }
      }
      if (live) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] *= p.scale;
        store_vec<T, VEC>(dx, r * p.dim + c, acc);
      }
    }
  }
  for (int i = 0; i < shared; ++i) {
    const int64_t r = i < s_hubs[1] ? s_hub[kHubList - 1 - i] : s_hub[i - s_hubs[1]];
    const int64_t lo = static_cast<int64_t>(indptr[r]), hi = static_cast<int64_t>(indptr[r + 1]);
    for (int64_t c0 = 0; c0 < p.dim; c0 += LPR * VEC) {
      const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
      const bool live = c < p.dim;
      float acc[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
      add_span(lo, hi, c, acc);   // (all groups have some of the edges)
      over_groups(acc);
      if (grp == 0 && live) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] *= p.scale;
        store_vec<T, VEC>(dx, r * p.dim + c, acc);
      }
    }
  }
}

// A workgroup for two rows per lane group, or, where rows have many edges, for sixteen edges per lane group (1 M edges of
// 16 fp32 into 4096 rows: 481 us with the 64 workgroups of the rows alone).
template <typename T, int VEC, typename I, bool EDATA>
static void launch_source_sum(SourceSumParams p, int64_t num_edges, hipStream_t st) {
  const int64_t per_row = ceil_div(p.dim, VEC);
#define APT_SOURCE_SUM(LPR)                                                                                        \
  do {                                                                                                            \
    constexpr int64_t groups = kAggBlock / LPR;                                                                    \
    const int64_t blocks = even_grid(std::max(ceil_div(p.num_src, kHubList),                                      \
                                              std::min<int64_t>(std::max(ceil_div(p.num_src, groups * 2),         \
                                                                         std::min(p.num_src, num_edges / (groups * kHubEdges))), \
                                                                kSourceBlocks)));                                 \
    const int64_t chunks = p.lng.slots > 0 ? std::min<int64_t>(long_chunks(num_edges), kLongBlocks) : 0;          \
    p.row_blocks = static_cast<uint32_t>(blocks);                                                                 \
    const dim3 grid(static_cast<unsigned>(blocks + chunks)), block(kAggBlock);                                    \
    if (chunks > 0) hipLaunchKernelGGL((source_sum_kernel<T, VEC, LPR, I, EDATA, true>), grid, block, 0, st, p);  \
    else hipLaunchKernelGGL((source_sum_kernel<T, VEC, LPR, I, EDATA, false>), grid, block, 0, st, p);            \
  } while (0)
  if (per_row <= 8) APT_SOURCE_SUM(8);
  else if (per_row <= 16) APT_SOURCE_SUM(16);
  else if (per_row <= 32) APT_SOURCE_SUM(32);
  else APT_SOURCE_SUM(64);
#undef APT_SOURCE_SUM
}

template <typename I, bool EDATA>
static int source_sum(SourceSumParams p, int64_t num_edges, int elem_size, hipStream_t st) {
  if (p.num_dst == 0) {   // no edge counts then, but entry 0 is read in the place of a missing one
    p.dz = p.dx;
    p.dst_scale = nullptr;
  }
  if (num_edges == 0) {
    p.via = nullptr;
    if (p.index != nullptr) p.index = p.indptr;
  }
  const bool aligned = ((reinterpret_cast<uintptr_t>(p.dz) | reinterpret_cast<uintptr_t>(p.dx) |
                         reinterpret_cast<uintptr_t>(p.edata)) & 15) == 0;
  if (elem_size == 4) {
    if (aligned && p.dim % 4 == 0) launch_source_sum<float, 4, I, EDATA>(p, num_edges, st);
    else launch_source_sum<float, 1, I, EDATA>(p, num_edges, st);
  } else {
    if (aligned && p.dim % 8 == 0) launch_source_sum<uint16_t, 8, I, EDATA>(p, num_edges, st);
    else if (aligned && p.dim % 4 == 0) launch_source_sum<uint16_t, 4, I, EDATA>(p, num_edges, st);
    else launch_source_sum<uint16_t, 1, I, EDATA>(p, num_edges, st);
  }
  APT_LAUNCH_CHECK("source_sum_kernel");
  return APT_OK;
}

// ------------------------------------------------------------------ long rows of given offsets
// A wavefront per slot of the table: the last row that begins in the slot's edges is the only one that can be
// long (a long row reaches beyond them).  Offsets are searched 64 at a time.
template <typename I>
__global__ __launch_bounds__(kAggBlock) void find_long_rows_kernel(const I* __restrict__ indptr, int64_t num_rows, LongRows l) {
  const int lane = threadIdx.x % kWave;
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * kAggWaves + threadIdx.x / kWave;
  if (slot >= l.slots) return;   // wave-uniform
  const int64_t from = slot * l.longer, to = from + l.longer;
  int64_t lo = 0, len = num_rows;   // rows that begin before `to`: lo + some of the next len
  while (len > 0) {
    const int64_t step = (len + kWave - 1) / kWave;
    const int64_t at = lo + lane * step + step - 1;   // the last row of the lane's stretch
    const uint64_t below = ballot(at < lo + len && static_cast<int64_t>(indptr[min(at, num_rows - 1)]) < to);
    const int64_t whole = __popcll(below);            // (offsets do not decrease: the lanes below are the first ones)
    const int64_t end = lo + len;
    lo += whole * step;
    len = min(step - 1, end - lo);
  }
  uint32_t found = 0;
  if (lo > 0) {
    const int64_t first = static_cast<int64_t>(indptr[lo - 1]), last = static_cast<int64_t>(indptr[lo]);
    if (first >= from && last - first > l.longer) found = static_cast<uint32_t>(lo);   // row lo - 1, plus one
  }
  if (lane == 0) {
    l.row[slot] = found;
    l.arrived[slot] = 0;
  }
}

// ------------------------------------------------------------------ sums over a COO
// The edges of a COO by absolute output row (`key`) and input row, whatever segments they come in, and whether the
// keys are non-decreasing.
struct CooParams {
  const int64_t* row;
  const int64_t* col;
  int64_t num_edges;
  const int64_t* coo_off;   // [num_seg + 1]
  const int64_t* in_off;    // [num_seg] or NULL
  const int64_t* out_off;   // [num_seg] or NULL
  int num_seg;
  int64_t* keys;
  int64_t* sources;
  int64_t* grouped;         // [0]: 1 on entry; [2]: 0 on entry, 1 if grouped keys may have a long row
  int64_t half;             // half of the edges that make a row long
};
constexpr int kCooSegments = APT_MAX_BUCKETS + 1;

__global__ void coo_grouped_init_kernel(int64_t* grouped, const int64_t* last_offset, int64_t* num_out) {
  grouped[0] = 1;
  grouped[2] = 0;
  *num_out = last_offset != nullptr ? *last_offset : 0;
}

__global__ __launch_bounds__(kAggBlock) void coo_prepare_kernel(CooParams p) {
  __shared__ int64_t s_off[kCooSegments + 1], s_in[kCooSegments], s_out[kCooSegments];
  if (static_cast<int>(threadIdx.x) <= p.num_seg) s_off[threadIdx.x] = p.coo_off[threadIdx.x];
  if (static_cast<int>(threadIdx.x) < p.num_seg) {
    s_in[threadIdx.x] = p.in_off != nullptr ? p.in_off[threadIdx.x] : 0;
    s_out[threadIdx.x] = p.out_off != nullptr ? p.out_off[threadIdx.x] : 0;
  }
  __syncthreads();
  auto segment = [&](int64_t e) {   // last k with coo_off[k] <= e (reference: cub::UpperBound - 1)
    int k = 0;
    while (k + 1 < p.num_seg && s_off[k + 1] <= e) ++k;
    return k;
  };
  bool bad = false, lengthy = false;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kAggBlock + threadIdx.x; e < p.num_edges;
       e += static_cast<int64_t>(gridDim.x) * kAggBlock) {
    const int k = segment(e);
    const int64_t key = s_out[k] + p.col[e];
    p.keys[e] = key;
    p.sources[e] = s_in[k] + p.row[e];
    if (e + 1 < p.num_edges) {
      const int q = segment(e + 1);
      bad |= key > s_out[q] + p.col[e + 1];
    }
    // a long row of equal keys: a multiple of half its length at least, and the key half that further on, are both in it
    if (e % p.half == 0 && e + p.half < p.num_edges) lengthy |= key == s_out[segment(e + p.half)] + p.col[e + p.half];
  }
  if (bad) p.grouped[0] = 0;
  if (lengthy) p.grouped[2] = 1;
}

// Offsets of the rows in non-decreasing keys: position e, where the key before it is kp and its own k, is the offset
// of the rows in (kp, k]; a long stretch of rows without edges is filled by the whole wavefront.
__global__ __launch_bounds__(kAggBlock) void coo_offsets_kernel(const int64_t* __restrict__ keys, int64_t n,
                                                                int64_t num_rows, uint32_t* __restrict__ indptr) {
  constexpr int kShortGap = 4;
  const int lane = threadIdx.x % kWave;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * kAggBlock + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kAggBlock;
  auto clamp = [&](int64_t k) { return k < -1 ? -1 : k > num_rows ? num_rows : k; };
  for (int64_t e0 = tid - lane; e0 < n; e0 += stride) {   // wave-uniform
    const int64_t e = e0 + lane;
    int64_t k = -1, kp = -1;
    if (e < n) {
      k = clamp(keys[e]);
      if (e > 0) kp = clamp(keys[e - 1]);
    }
    const int64_t gap = k - kp;
    if (gap > 0 && gap <= kShortGap)
      for (int64_t t = kp + 1; t <= k; ++t) indptr[t] = static_cast<uint32_t>(e);
    uint64_t wide = ballot(gap > kShortGap);
    while (wide != 0) {
      const int src = __ffsll(static_cast<long long>(wide)) - 1;
      wide &= wide - 1;
      const int64_t a = __shfl(kp, src, kWave) + 1, b = __shfl(k, src, kWave);
      for (int64_t t = a + lane; t <= b; t += kWave) indptr[t] = static_cast<uint32_t>(e0 + src);
    }
  }
  const int64_t last = n > 0 ? clamp(keys[n - 1]) : -1;
  for (int64_t t = last + 1 + tid; t <= num_rows; t += stride) indptr[t] = static_cast<uint32_t>(n);
}

static size_t coo_align(size_t x) { return (x + 255) / 256 * 256; }

}  // namespace apt

extern "C" int apt_coo_prepare(const int64_t* coo_row, const int64_t* coo_col, int64_t num_edges, const int64_t* coo_offset,
                               const int64_t* input_offset, const int64_t* output_offset, int num_segments,
                               const int64_t* last_offset, int64_t* keys, int64_t* sources, int64_t* result, void* stream) {
  using namespace apt;
  APT_REQUIRE(num_edges >= 0 && result != nullptr, APT_EINVAL, "apt_coo_prepare: bad arguments");
  APT_REQUIRE(num_segments >= 1 && num_segments < kCooSegments, APT_ELIMIT, "apt_coo_prepare: %d segments outside [1, %d]",
              num_segments, kCooSegments - 1);
  APT_REQUIRE(num_edges == 0 || (coo_row != nullptr && coo_col != nullptr && coo_offset != nullptr && keys != nullptr &&
                                 sources != nullptr),
              APT_EINVAL, "apt_coo_prepare: a tensor is NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(coo_grouped_init_kernel, dim3(1), dim3(1), 0, st, result, last_offset, result + 1);
  APT_LAUNCH_CHECK("coo_grouped_init_kernel");
  if (num_edges == 0) return APT_OK;
  const CooParams p{coo_row, coo_col, num_edges, coo_offset, input_offset, output_offset, num_segments, keys, sources, result,
                    long_from(num_edges) / 2};
  hipLaunchKernelGGL(coo_prepare_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(num_edges, kAggBlock), 4096))),
                     dim3(kAggBlock), 0, st, p);
  APT_LAUNCH_CHECK("coo_prepare_kernel");
  return APT_OK;
}

namespace apt {
// A sum's scratch: the table of its long rows, if it makes one itself, and their chunks' sums.
static size_t long_table_bytes(int64_t num_edges) { return coo_align(sizeof(uint32_t) * 2 * long_slots(num_edges)); }
static size_t long_part_bytes(int64_t num_edges, int64_t width) { return coo_align(sizeof(float) * long_chunks(num_edges) * width); }

template <typename I>
static int find_long_rows(const void* indptr, int64_t num_rows, const LongRows& l, hipStream_t st) {
  if (l.slots == 0) return APT_OK;
  hipLaunchKernelGGL(find_long_rows_kernel<I>, dim3(static_cast<unsigned>(ceil_div(l.slots, kAggWaves))), dim3(kAggBlock), 0, st,
                     static_cast<const I*>(indptr), num_rows, l);
  APT_LAUNCH_CHECK("find_long_rows_kernel");
  return APT_OK;
}
}  // namespace apt

extern "C" size_t apt_long_rows_bytes(int64_t num_edges) {
  return num_edges < 0 || num_edges > 0x7fffffffLL ? 0 : apt::long_table_bytes(num_edges);
}

extern "C" int apt_find_long_rows(const void* indptr, int index_bytes, int64_t num_src, int64_t num_edges, void* long_table,
                                  void* stream) {
  using namespace apt;
  APT_REQUIRE(num_src >= 0 && num_src <= 0x7fffffffLL && num_edges >= 0 && num_edges <= 0x7fffffffLL, APT_ELIMIT,
              "apt_find_long_rows: sizes out of range (num_src %lld, edges %lld)", (long long)num_src, (long long)num_edges);
  APT_REQUIRE(index_bytes == 4 || index_bytes == 8, APT_EINVAL, "apt_find_long_rows: index_bytes %d", index_bytes);
  if (long_slots(num_edges) == 0) return APT_OK;
  APT_REQUIRE(indptr != nullptr && long_table != nullptr, APT_EINVAL, "apt_find_long_rows: a tensor is NULL");
  const LongRows l = long_rows(long_table, num_edges, nullptr);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return index_bytes == 8 ? find_long_rows<int64_t>(indptr, num_src, l, st) : find_long_rows<uint32_t>(indptr, num_src, l, st);
}

extern "C" size_t apt_coo_sum_workspace_bytes(int64_t num_edges, int64_t num_out_rows, int grouped, int has_long, int64_t dim) {
  using namespace apt;
  if (num_edges < 0 || num_edges > 0x7fffffffLL || num_out_rows < 0 || num_out_rows > 0x7fffffffLL || dim <= 0) return 0;
  size_t offsets = coo_align(sizeof(uint32_t) * (num_out_rows + 1));
  if (grouped == 0 || has_long != 0) offsets += long_table_bytes(num_edges) + long_part_bytes(num_edges, dim);
  if (grouped != 0) return offsets;
  const size_t order = apt_block_transpose_workspace_bytes(num_edges, 1, num_out_rows);
  return order == 0 ? 0 : offsets + coo_align(sizeof(uint32_t) * (num_edges + 1)) + order;
}

extern "C" int apt_coo_sum(int mode, const int64_t* keys, const int64_t* sources, int64_t num_edges, int grouped, int has_long,
                           const void* input, int64_t num_in_rows, const void* edata, int64_t dim, int elem_size, void* out,
                           int64_t num_out_rows, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(mode >= 0 && mode <= 2, APT_EINVAL, "apt_coo_sum: mode %d (0 copy_u, 1 copy_e, 2 u_mul_e)", mode);
  APT_REQUIRE(num_edges >= 0 && num_in_rows >= 0 && num_out_rows >= 0 && dim > 0, APT_EINVAL,
              "apt_coo_sum: bad shape (E %lld, rows %lld -> %lld, dim %lld)", (long long)num_edges, (long long)num_in_rows,
              (long long)num_out_rows, (long long)dim);
  APT_REQUIRE(elem_size == 2 || elem_size == 4, APT_EINVAL, "apt_coo_sum: elem_size %d (4 = fp32, 2 = bf16)", elem_size);
  if (num_out_rows == 0) return APT_OK;
  const size_t need = apt_coo_sum_workspace_bytes(num_edges, num_out_rows, grouped, has_long, dim);
  APT_REQUIRE(need > 0, APT_ELIMIT, "apt_coo_sum: %lld edges or %lld rows out of range", (long long)num_edges,
              (long long)num_out_rows);
  APT_REQUIRE(out != nullptr && (num_edges == 0 || (keys != nullptr && sources != nullptr && input != nullptr)) &&
                  (mode != 2 || edata != nullptr || num_edges == 0),
              APT_EINVAL, "apt_coo_sum: a tensor is NULL");
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 255) == 0,
              APT_EWORKSPACE, "apt_coo_sum: workspace too small or not 256-byte aligned (see apt_coo_sum_workspace_bytes)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  uint32_t* indptr = reinterpret_cast<uint32_t*>(ws);
  ws += coo_align(sizeof(uint32_t) * (num_out_rows + 1));
  LongRows lng{};
  if (grouped == 0 || has_long != 0) {
    lng = long_rows(ws, num_edges, reinterpret_cast<float*>(ws + long_table_bytes(num_edges)));
    ws += long_table_bytes(num_edges) + long_part_bytes(num_edges, dim);
  }
  uint32_t* order = nullptr;
  if (grouped != 0) {
    const int64_t work = std::max(num_edges, num_out_rows + 1);
    hipLaunchKernelGGL(coo_offsets_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(work, kAggBlock), 4096))),
                       dim3(kAggBlock), 0, st, keys, num_edges, num_out_rows, indptr);
    APT_LAUNCH_CHECK("coo_offsets_kernel");
    if (const int rc = find_long_rows<uint32_t>(indptr, num_out_rows, lng, st)) return rc;
  } else {
    order = reinterpret_cast<uint32_t*>(ws);
    ws += coo_align(sizeof(uint32_t) * (num_edges + 1));
    const size_t left = workspace_bytes - static_cast<size_t>(ws - static_cast<char*>(workspace));
    if (const int rc = apt_block_transpose(keys, num_edges, 1, num_out_rows, indptr, order, lng.row, ws, left, stream)) return rc;
  }
  SourceSumParams p{};
  p.scale = 1.f;
  p.indptr = indptr;
  p.index = order;
  p.fanout = 1;
  p.via = mode == 1 ? nullptr : sources;
  p.edata = mode == 2 ? edata : nullptr;
  p.dz = input;
  p.num_dst = mode == 1 ? num_edges : num_in_rows;
  p.dim = dim;
  p.num_src = num_out_rows;
  p.dx = out;
  p.lng = lng;
  return mode == 2 ? source_sum<uint32_t, true>(p, num_edges, elem_size, st)
                   : source_sum<uint32_t, false>(p, num_edges, elem_size, st);
}

extern "C" size_t apt_block_aggregate_backward_workspace_bytes(int64_t num_edges, int64_t dim) {
  return num_edges < 0 || num_edges > 0x7fffffffLL || dim <= 0 ? 0 : apt::long_part_bytes(num_edges, dim);
}

extern "C" int apt_block_aggregate_backward(const void* indptr, const void* index, int index_bytes, int fanout,
                                            int64_t num_src, int64_t num_edges, void* long_table, const float* dst_scale,
                                            float scale, const void* dz, int64_t num_dst, int64_t dim, int elem_size, void* dx,
                                            void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(num_src >= 0 && num_src <= 0x7fffffffLL && num_edges >= 0 && num_edges <= 0x7fffffffLL && num_dst >= 0 && dim > 0,
              APT_EINVAL, "apt_block_aggregate_backward: bad shape (num_src %lld, edges %lld, num_dst %lld, dim %lld)",
              (long long)num_src, (long long)num_edges, (long long)num_dst, (long long)dim);
  APT_REQUIRE(elem_size == 2 || elem_size == 4, APT_EINVAL,
              "apt_block_aggregate_backward: elem_size %d (4 = fp32, 2 = bf16)", elem_size);
  APT_REQUIRE(index_bytes == 8 || (index_bytes == 4 && fanout > 0), APT_EINVAL,
              "apt_block_aggregate_backward: index_bytes %d (8 = destinations, 4 = slots, with the fanout)", index_bytes);
  if (num_src == 0) return APT_OK;
  APT_REQUIRE(indptr != nullptr && dx != nullptr && (num_dst == 0 || dz != nullptr) && (num_edges == 0 || index != nullptr),
              APT_EINVAL, "apt_block_aggregate_backward: a tensor is NULL");
  const size_t need = long_table == nullptr ? 0 : apt_block_aggregate_backward_workspace_bytes(num_edges, dim);
  APT_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0),
              APT_EWORKSPACE, "apt_block_aggregate_backward: workspace too small or not 16-byte aligned "
                              "(see apt_block_aggregate_backward_workspace_bytes)");
  SourceSumParams p{};
  p.indptr = indptr;
  p.index = index != nullptr ? index : indptr;   // (no edge: never read)
  p.fanout = static_cast<uint32_t>(fanout);
  p.dst_scale = dst_scale;
  p.scale = scale;
  p.dz = dz;
  p.num_dst = num_dst;
  p.dim = dim;
  p.num_src = num_src;
  p.dx = dx;
  p.lng = long_rows(long_table, num_edges, static_cast<float*>(workspace));
  hipStream_t st = static_cast<hipStream_t>(stream);
  return index_bytes == 8 ? source_sum<int64_t, false>(p, num_edges, elem_size, st)
                          : source_sum<uint32_t, false>(p, num_edges, elem_size, st);
}

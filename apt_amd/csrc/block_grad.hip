// Source side of a block's aggregation: dx[s, :] = sum over the edges s -> d of w(e) * dz[d, :], the gradient of the
// block sum / mean (and, weighted per edge and head, of the GAT aggregation) towards its input.
//
// A lane group owns a source row, so every row is written once, in its own type, whole and in a fixed order: no
// zero-fill, no atomics, no fp32 copy of a bf16 result.  Nearly all sources of a sampled block have one or two edges;
// two rows per group are in flight.  The few hubs (hundreds of edges) would each occupy one group for the length of
// the launch: rows longer than kHubEdges are put aside and added up by all groups of the workgroup afterwards.  Hubs
// have neighbouring ids (the relabel numbers nodes by first occurrence), so a workgroup's rows are taken a grid apart.
#include <algorithm>

#include "common.hpp"
#include "feature_rows.hpp"

namespace apt {

constexpr int kHubEdges = 32;
constexpr int kHubList = 1024;             // rows of a workgroup at the most, so its list of hubs never overflows
constexpr int kSourceBlocks = 2048;

struct SourceSumParams {
  const void* indptr;      // offsets of the sources in `index`
  const void* index;       // per edge: its destination, or its slot (fanout > 0: destination = slot / fanout)
  uint32_t fanout;
  const float* dst_scale;  // per destination, or NULL
  const void* dz;          // [num_dst, dim]
  int64_t num_dst;
  int64_t dim;
  int64_t num_src;
  void* dx;                // [num_src, dim]
};

// I: int64_t = a block's CSR (offsets, destinations), uint32_t = apt_block_transpose (offsets, slots).
template <typename T, int VEC, int LPR, typename I>
__global__ __launch_bounds__(kAggBlock) void source_sum_kernel(SourceSumParams p) {
  constexpr int kGroups = kAggBlock / LPR;
  constexpr int kRows = 2;
  constexpr int kUnroll = 4;
  __shared__ int s_hub[kHubList];
  __shared__ int s_hubs;
  __shared__ float s_sum[kGroups][LPR * VEC];
  const int grp = threadIdx.x / LPR, l = threadIdx.x % LPR;
  const I* indptr = static_cast<const I*>(p.indptr);
  const I* index = static_cast<const I*>(p.index);
  const T* dz = static_cast<const T*>(p.dz);
  T* dx = static_cast<T*>(p.dx);
  if (threadIdx.x == 0) s_hubs = 0;
  __syncthreads();
  auto destination = [&](I i) -> int64_t {
    const int64_t d = sizeof(I) == 4 ? static_cast<int64_t>(static_cast<uint32_t>(i) / p.fanout) : static_cast<int64_t>(i);
    return d >= 0 && d < p.num_dst ? d : -1;
  };
  // acc += the rows of up to LPR edges whose destinations the group's lanes hold (lane j: edge j)
  auto add_edges = [&](int64_t my_dst, float my_scale, int n, int64_t c, bool live, float (&acc)[VEC]) {
    for (int e0 = 0; e0 < n; e0 += kUnroll) {
      float v[kUnroll][VEC];
      float w[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) v[u][k] = 0.f;
        w[u] = 0.f;
        if (e0 + u < n) {
          const int64_t d = __shfl(my_dst, e0 + u, LPR);
          w[u] = __shfl(my_scale, e0 + u, LPR);
          if (d >= 0 && live) load_vec<T, VEC>(dz, d * p.dim + c, v[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] += w[u] * v[u][k];
    }
  };
  const int64_t row_groups = static_cast<int64_t>(gridDim.x) * kGroups;
  for (int64_t r0 = static_cast<int64_t>(grp) * gridDim.x + blockIdx.x; r0 < p.num_src; r0 += kRows * row_groups) {
    int64_t lo[kRows];
    int n[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const int64_t r = r0 + q * row_groups;
      lo[q] = 0;
      n[q] = 0;
      if (r < p.num_src) {
        lo[q] = static_cast<int64_t>(indptr[r]);
        n[q] = static_cast<int>(static_cast<int64_t>(indptr[r + 1]) - lo[q]);
      }
    }
    int64_t dst[kRows];
    float scale[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) dst[q] = l < n[q] && n[q] <= kHubEdges ? destination(index[lo[q] + l]) : -1;
#pragma unroll
    for (int q = 0; q < kRows; ++q) scale[q] = p.dst_scale != nullptr && dst[q] >= 0 ? p.dst_scale[dst[q]] : 1.f;
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
        add_edges(dst[q], scale[q], min(n[q], LPR), c, live, acc);
        for (int e = LPR; e < n[q]; e += LPR) {   // LPR < kHubEdges only
          const int64_t d = e + l < n[q] ? destination(index[lo[q] + e + l]) : -1;
          const float s = p.dst_scale != nullptr && d >= 0 ? p.dst_scale[d] : 1.f;
          add_edges(d, s, min(n[q] - e, LPR), c, live, acc);
        }
        if (live) store_vec<T, VEC>(dx, r * p.dim + c, acc);
      }
    }
#pragma unroll
    for (int q = 0; q < kRows; ++q)
      if (n[q] > kHubEdges && l == 0) s_hub[atomicAdd(&s_hubs, 1)] = static_cast<int>(r0 + q * row_groups);
  }
  __syncthreads();
  const int hubs = s_hubs;
  for (int i = 0; i < hubs; ++i) {   // (in any order: every hub is summed on its own)
    const int64_t r = s_hub[i];
    const int64_t lo = static_cast<int64_t>(indptr[r]), hi = static_cast<int64_t>(indptr[r + 1]);
    for (int64_t c0 = 0; c0 < p.dim; c0 += LPR * VEC) {
      const int64_t c = c0 + static_cast<int64_t>(l) * VEC;
      const bool live = c < p.dim;
      float acc[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
      for (int64_t e = lo + grp * LPR; e < hi; e += kAggBlock) {
        const int64_t d = e + l < hi ? destination(index[e + l]) : -1;
        const float s = p.dst_scale != nullptr && d >= 0 ? p.dst_scale[d] : 1.f;
        add_edges(d, s, static_cast<int>(min(hi - e, static_cast<int64_t>(LPR))), c, live, acc);
      }
#pragma unroll
      for (int k = 0; k < VEC; ++k) s_sum[grp][l * VEC + k] = acc[k];
      __syncthreads();
      if (grp == 0 && live) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          float sum = 0.f;
#pragma unroll 1
          for (int g = 0; g < kGroups; ++g) sum += s_sum[g][l * VEC + k];
          acc[k] = sum;
        }
        store_vec<T, VEC>(dx, r * p.dim + c, acc);
      }
      __syncthreads();
    }
  }
}

template <typename T, int VEC, typename I>
static void launch_source_sum(const SourceSumParams& p, hipStream_t st) {
  const int64_t per_row = ceil_div(p.dim, VEC);
#define APT_SOURCE_SUM(LPR)                                                                                        \
  do {                                                                                                            \
    constexpr int64_t groups = kAggBlock / LPR;                                                                    \
    const int64_t blocks = std::max(ceil_div(p.num_src, kHubList),                                                \
                                    std::min<int64_t>(ceil_div(p.num_src, groups * 2), kSourceBlocks));           \
    hipLaunchKernelGGL((source_sum_kernel<T, VEC, LPR, I>), dim3(static_cast<unsigned>(blocks)), dim3(kAggBlock), 0, \
                       st, p);                                                                                    \
  } while (0)
  if (per_row <= 8) APT_SOURCE_SUM(8);
  else if (per_row <= 16) APT_SOURCE_SUM(16);
  else if (per_row <= 32) APT_SOURCE_SUM(32);
  else APT_SOURCE_SUM(64);
#undef APT_SOURCE_SUM
}

template <typename I>
static int source_sum(const SourceSumParams& p, int elem_size, hipStream_t st) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(p.dz) | reinterpret_cast<uintptr_t>(p.dx)) & 15) == 0;
  if (elem_size == 4) {
    if (aligned && p.dim % 4 == 0) launch_source_sum<float, 4, I>(p, st);
    else launch_source_sum<float, 1, I>(p, st);
  } else {
    if (aligned && p.dim % 8 == 0) launch_source_sum<uint16_t, 8, I>(p, st);
    else if (aligned && p.dim % 4 == 0) launch_source_sum<uint16_t, 4, I>(p, st);
    else launch_source_sum<uint16_t, 1, I>(p, st);
  }
  APT_LAUNCH_CHECK("source_sum_kernel");
  return APT_OK;
}

}  // namespace apt

extern "C" int apt_block_aggregate_backward(const void* indptr, const void* index, int index_bytes, int fanout,
                                            int64_t num_src, const float* dst_scale, const void* dz, int64_t num_dst,
                                            int64_t dim, int elem_size, void* dx, void* stream) {
  using namespace apt;
  APT_REQUIRE(num_src >= 0 && num_src <= 0x7fffffffLL && num_dst >= 0 && dim > 0, APT_EINVAL,
              "apt_block_aggregate_backward: bad shape (num_src %lld, num_dst %lld, dim %lld)", (long long)num_src,
              (long long)num_dst, (long long)dim);
  APT_REQUIRE(elem_size == 2 || elem_size == 4, APT_EINVAL,
              "apt_block_aggregate_backward: elem_size %d (4 = fp32, 2 = bf16)", elem_size);
  APT_REQUIRE(index_bytes == 8 || (index_bytes == 4 && fanout > 0), APT_EINVAL,
              "apt_block_aggregate_backward: index_bytes %d (8 = destinations, 4 = slots, with the fanout)", index_bytes);
  if (num_src == 0) return APT_OK;
  APT_REQUIRE(indptr != nullptr && dx != nullptr && (num_dst == 0 || (index != nullptr && dz != nullptr)), APT_EINVAL,
              "apt_block_aggregate_backward: a tensor is NULL");
  SourceSumParams p;
  p.indptr = indptr;
  p.index = index;
  p.fanout = static_cast<uint32_t>(fanout);
  p.dst_scale = dst_scale;
  p.dz = dz;
  p.num_dst = num_dst;
  p.dim = dim;
  p.num_src = num_src;
  p.dx = dx;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return index_bytes == 8 ? source_sum<int64_t>(p, elem_size, st) : source_sum<uint32_t>(p, elem_size, st);
}

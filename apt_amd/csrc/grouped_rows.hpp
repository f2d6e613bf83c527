// How the rows of a sum over grouped edges are dealt to lane groups (block_grad.hip, gat_layer.hip).
#pragma once

#include "common.hpp"

namespace apt {

// First row of a lane group.  The groups that work side by side on one XCD (workgroups eight apart) take 64 neighbouring
// rows: the relabel numbers sources by their first destination, so rows next to each other read the same rows of dz, and
// that XCD's L2 has them.  (num_src rows are taken a grid apart: hubs have neighbouring ids too.)
constexpr int kSlab = 64;
template <int GROUPS> __host__ __device__ constexpr int slab_blocks() { return kSlab / GROUPS; }
template <int GROUPS> __device__ __forceinline__ int64_t group_row(int grp, uint32_t blocks) {   // blocks: of the rows
  const uint32_t per = 8 * slab_blocks<GROUPS>();
  const uint32_t whole = blocks / per * per, b = blockIdx.x;
  if (b >= whole) return static_cast<int64_t>(b) * GROUPS + grp;   // what is left of the grid: in a row
  const uint32_t xcd = b % 8, j = b / 8;                           // the j-th workgroup of the XCD
  return (static_cast<int64_t>(j / slab_blocks<GROUPS>()) * 8 + xcd) * kSlab + grp * slab_blocks<GROUPS>() + j % slab_blocks<GROUPS>();
}

// Edges of a hub that one lane group adds up by itself: with 128 instead of 32 a hub of 100 edges is the tail of a launch
// (54 k sources, 256 fp32: 36 us instead of 27), with 32 instead of 128 the 32 groups of a workgroup meet for a few edges
// each (238 k sources, 64 bf16, with the ordering: 204 us instead of 145).
template <int LPR> constexpr int hub_shared() { return LPR <= 8 ? 128 : 32; }

}  // namespace apt

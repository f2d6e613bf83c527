// How the rows of a sum over grouped edges are dealt to lane groups (block_grad.hip, gat_layer.hip).
#pragma once

#include "common.hpp"

namespace apt {

// Scalar registers of a kernel that is to have eight wavefronts on a SIMD: with 82 and more (for which the compiler still
// tells eight) a launch of 2048 workgroups takes a second turn for the last of them.  500 k rows of 47 fp32: 152 us with
// 82..100, 101 with 80; with 4096 workgroups a tail costs half as much.
constexpr int kFullSgprs = 80;

// First row of a lane group.  The groups that work side by side on one XCD (workgroups eight apart) take 64 neighbouring
// rows: the relabel numbers sources by their first destination, so rows next to each other read the same rows of dz, and
// that XCD's L2 has them.  Each of the 64 is another workgroup's, and the next 64 are another XCD's: hubs have neighbouring
// ids too.  (Four neighbours to a workgroup, whose first cache they would share: 38 instead of 41 us for 124 k sampled rows of
// 4 x 64 bf16, but 223 instead of 92 for 240 k rows of 47 fp32 whose first thousands are hubs.)  A grid that does not come
// out even (or has no 64 workgroups on an XCD) takes its rows one by one.
constexpr int kSlab = 64;
static int64_t even_grid(int64_t blocks) { return blocks < 8 * kSlab ? blocks : ceil_div(blocks, 8 * kSlab) * (8 * kSlab); }
template <int GROUPS> __device__ __forceinline__ int64_t group_row(int grp, uint32_t blocks) {   // blocks: of the rows
  const uint32_t b = blockIdx.x;
  if (blocks % (8 * kSlab) != 0) return static_cast<int64_t>(grp) * blocks + b;
  const uint32_t xcd = b % 8, q = static_cast<uint32_t>(grp) * (blocks / 8) + b / 8;   // the q-th group of the XCD
  return (static_cast<int64_t>(q / kSlab) * 8 + xcd) * kSlab + q % kSlab;
}

// Hubs that lane groups add up on their own: those of at most so many edges, if a workgroup has so many of them.  A hub that
// all groups of a workgroup add up costs them a meeting (two barriers and a sum), one that a group adds up alone is the tail
// of a launch.  30 k rows of 25 edges, 47 / 256 bf16: 64 / 60 us, with 32 instead of 64 edges 67 / 70; 238 k sampled
// sources, 64 bf16, 32 instead of 128 edges for the narrowest groups: 204 us instead of 145.  With hubs for a quarter / an
// eighth / a sixteenth of the groups: 2 k skewed rows of 25 k edges, 16 bf16, 95 / 41 / 42 us; 8 k rows of 125 edges, 16 fp32,
// 63 / 63 / 80.  A workgroup's only hub is always all groups' (256 x 10 skewed edges into 2 k rows of 100 fp32: 6.4 us, 12.2 alone).
template <int LPR> constexpr int hub_shared() { return LPR <= 8 ? 128 : LPR >= 32 ? 64 : 32; }
template <int GROUPS> constexpr int hubs_apiece() { return GROUPS > 16 ? GROUPS / 8 : 2; }

}  // namespace apt

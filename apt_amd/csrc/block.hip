// Sparse formats of a sampled block.
//
// A hop leaves a fixed-stride block: relabeled[d * fanout + k] is the k-th
// source of destination d, -1 where d has fewer than fanout neighbours.  The
// reference hands (row, col) to DGL, which materialises COO, CSR and CSC
// (python/npc/sampler.py:59-69,76-91; create_block_from_csc :44-56 takes a CSC
// directly).  Here the three formats are emitted on the GPU, with device-side
// sizes and no host round trip:
//   COO  edges in destination-major order: row[e] = source, col[e] = destination
//   CSC  csc_indptr over destinations; its indices are COO row, edge ids 0..E-1
//   CSR  csr_indptr over sources, csr_indices = destination, csr_eids = COO
//        position, edges of one source in increasing edge id
// COO/CSC are a stream compaction (count per tile -> place).  CSR of the blocks a
// sampler makes is a partition by source range carried along with that
// compaction, then a counting sort of every range in one workgroup (below, "CSR by
// source ranges"): four launches for all three formats.  Blocks of more than 6 M
// sources, 8 M slots or 2 M destinations, and blocks of very few sources, take a stable
// least-significant-digit radix sort of (source, edge id) by source, 8 bits per pass (histogram per tile ->
// scatter).  Everywhere a workgroup ranks its tile with wave ballots, so equal keys
// keep their order and the result is reproducible (no atomic tickets).  A block
// of a mini-batch has few tiles, so the place and scatter workgroups add up the
// counts of the tiles before them themselves (a few KB from L2) instead of waiting
// for a scan kernel: every launch saved is worth more than the arithmetic here.
// Large inputs take separate scan launches.
#include <algorithm>

#include "common.hpp"
#include "long_rows.hpp"

namespace apt {

constexpr int kFmtBlock = 256;
constexpr int kFmtWaves = kFmtBlock / kWave;
constexpr int kCompactIters = 8;
constexpr int kCompactTile = kFmtBlock * kCompactIters;  // slots per workgroup
constexpr int kSortBlock = kFmtBlock;
constexpr int kSortWaves = kSortBlock / kWave;
constexpr int kSortRounds = 16;
constexpr int kSortWaveItems = kWave * kSortRounds;       // consecutive items of one wave
constexpr int kSortTile = kSortWaveItems * kSortWaves;    // items per workgroup
constexpr int64_t kFusedCompactTiles = 8192;              // up to here a workgroup sums the tile counts itself
constexpr int64_t kFusedSortTiles = 32;
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;
static_assert(kRadix == kSortBlock, "one thread per digit");
constexpr int kScanPerThread = 16;
constexpr int kScanChunk = kFmtBlock * kScanPerThread;    // elements per workgroup of the scan

// ------------------------------------------------------------------ scan
// Exclusive prefix sum of a uint32 array in place, at most kScanChunk^2
// elements: chunk sums -> scan of the sums (one workgroup) -> rescan + offset.
__device__ __forceinline__ int64_t ceil_div_dev(int64_t a, int64_t b) { return (a + b - 1) / b; }

__device__ __forceinline__ uint32_t block_exclusive(uint32_t x, uint32_t* s_wave, uint32_t& all) {
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  uint32_t incl = x;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t y = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += y;
  }
  __syncthreads();  // s_wave may still be read by the previous call
  if (lane == kWave - 1) s_wave[wave] = incl;
  __syncthreads();
  uint32_t before = 0;
  all = 0;
#pragma unroll
  for (int w = 0; w < kFmtWaves; ++w) {
    const uint32_t c = s_wave[w];
    if (w < wave) before += c;
    all += c;
  }
  return before + incl - x;
}

__global__ __launch_bounds__(kFmtBlock) void scan_sums_kernel(const uint32_t* __restrict__ data, int64_t n,
                                                              uint32_t* __restrict__ sums) {
  __shared__ uint32_t s_wave[kFmtWaves];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanChunk;
  uint32_t acc = 0;
#pragma unroll
  for (int k = 0; k < kScanPerThread; ++k) {
    const int64_t i = base + k * kFmtBlock + threadIdx.x;
    if (i < n) acc += data[i];
  }
  uint32_t all;
  block_exclusive(acc, s_wave, all);
  if (threadIdx.x == 0) sums[blockIdx.x] = all;
}

// One workgroup: sums[0..m) -> exclusive prefix, m <= kScanChunk; the grand
// total goes to total_a / total_b (either may be NULL).
__global__ __launch_bounds__(kFmtBlock) void scan_top_kernel(uint32_t* sums, int64_t m, int64_t* total_a,
                                                             int64_t* total_b) {
  __shared__ uint32_t s_wave[kFmtWaves];
  uint32_t v[kScanPerThread];
  uint32_t acc = 0;
#pragma unroll
  for (int k = 0; k < kScanPerThread; ++k) {
    const int64_t i = static_cast<int64_t>(threadIdx.x) * kScanPerThread + k;
    v[k] = i < m ? sums[i] : 0u;
    acc += v[k];
  }
  uint32_t all;
  uint32_t run = block_exclusive(acc, s_wave, all);
#pragma unroll
  for (int k = 0; k < kScanPerThread; ++k) {
    const int64_t i = static_cast<int64_t>(threadIdx.x) * kScanPerThread + k;
    if (i < m) sums[i] = run;
    run += v[k];
  }
  if (threadIdx.x == 0) {
    if (total_a != nullptr) *total_a = all;
    if (total_b != nullptr) *total_b = all;
  }
}

__global__ __launch_bounds__(kFmtBlock) void scan_apply_kernel(uint32_t* data, int64_t n,
                                                               const uint32_t* __restrict__ sums) {
  __shared__ uint32_t s_wave[kFmtWaves];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanChunk +
                       static_cast<int64_t>(threadIdx.x) * kScanPerThread;
  uint32_t v[kScanPerThread];
  uint32_t acc = 0;
#pragma unroll
  for (int k = 0; k < kScanPerThread; ++k) {
    v[k] = base + k < n ? data[base + k] : 0u;
    acc += v[k];
  }
  uint32_t all;
  uint32_t run = sums[blockIdx.x] + block_exclusive(acc, s_wave, all);
#pragma unroll
  for (int k = 0; k < kScanPerThread; ++k) {
    if (base + k < n) data[base + k] = run;
    run += v[k];
  }
}

// data[0..n) -> exclusive prefix in place; sums: scratch of ceil(n / kScanChunk) entries.
static int exclusive_scan(uint32_t* data, int64_t n, uint32_t* sums, int64_t* total_a, int64_t* total_b,
                          hipStream_t st) {
  const int64_t chunks = ceil_div(n, kScanChunk);
  APT_REQUIRE(chunks <= kScanChunk, APT_ELIMIT, "block formats: %lld counters exceed the scan's range",
              static_cast<long long>(n));
  if (chunks <= 1) {
    hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(kFmtBlock), 0, st, data, n, total_a, total_b);
    APT_LAUNCH_CHECK("scan_top_kernel");
    return APT_OK;
  }
  hipLaunchKernelGGL(scan_sums_kernel, dim3(static_cast<unsigned>(chunks)), dim3(kFmtBlock), 0, st, data, n,
                     sums);
  APT_LAUNCH_CHECK("scan_sums_kernel");
  hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(kFmtBlock), 0, st, sums, chunks, total_a, total_b);
  APT_LAUNCH_CHECK("scan_top_kernel");
  hipLaunchKernelGGL(scan_apply_kernel, dim3(static_cast<unsigned>(chunks)), dim3(kFmtBlock), 0, st, data, n,
                     sums);
  APT_LAUNCH_CHECK("scan_apply_kernel");
  return APT_OK;
}

// ------------------------------------------------------------ COO + CSC
struct CompactParams {
  const int64_t* relabeled;
  int64_t num_dst;            // upper bound
  const int64_t* num_dst_dev;
  int fanout;
  uint32_t* tile_cnt;         // [tiles]; after a scan launch: the tile's first edge
  int64_t tiles;
  bool scanned;               // tile_cnt went through exclusive_scan
  int64_t* num_edges_dev;
  int64_t* coo_row;
  int64_t* coo_col;
  int64_t* csc_indptr;        // [num_dst + 1]
};

__global__ __launch_bounds__(kFmtBlock) void fmt_count_kernel(CompactParams p) {
  __shared__ uint32_t s_wave[kFmtWaves];
  const int64_t slots = actual_count(p.num_dst, p.num_dst_dev) * p.fanout;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kCompactTile;
  uint32_t c = 0;
#pragma unroll
  for (int it = 0; it < kCompactIters; ++it) {
    const int64_t s = base + it * kFmtBlock + threadIdx.x;
    if (s < slots && p.relabeled[s] >= 0) ++c;
  }
  uint32_t all;
  block_exclusive(c, s_wave, all);
  if (threadIdx.x == 0) p.tile_cnt[blockIdx.x] = all;
}

__global__ __launch_bounds__(kFmtBlock) void fmt_place_kernel(CompactParams p) {
  __shared__ uint32_t s_cnt[kCompactIters * kFmtWaves];
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const int64_t slots = actual_count(p.num_dst, p.num_dst_dev) * p.fanout;
  const int64_t upper = p.num_dst * p.fanout;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kCompactTile;
  int64_t v[kCompactIters];
  uint32_t below[kCompactIters];
#pragma unroll
  for (int it = 0; it < kCompactIters; ++it) {   // the tile's slots are all requested before the first is looked at
    const int64_t s = base + it * kFmtBlock + threadIdx.x;
    v[it] = s < slots ? p.relabeled[s] : -1;
  }
#pragma unroll
  for (int it = 0; it < kCompactIters; ++it) {
    const uint64_t m = ballot(v[it] >= 0);
    below[it] = rank_below(m);
    if (lane == 0) s_cnt[it * kFmtWaves + wave] = __popcll(m);
  }
  uint32_t first = 0;
  if (p.scanned) {
    first = p.tile_cnt[blockIdx.x];
  } else {
    // edges of the tiles before this one, and of all tiles
    __shared__ uint32_t s_wave[kFmtWaves];
    const int64_t active = ceil_div_dev(slots, kCompactTile);
    uint32_t before = 0, total = 0;
    for (int64_t t = threadIdx.x; t < active; t += kFmtBlock) {
      const uint32_t c = p.tile_cnt[t];
      total += c;
      if (t < blockIdx.x) before += c;
    }
    uint32_t all_before, all_total;
    block_exclusive(before, s_wave, all_before);
    block_exclusive(total, s_wave, all_total);
    first = all_before;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *p.num_edges_dev = all_total;
      p.csc_indptr[p.num_dst] = all_total;
    }
  }
  __syncthreads();
  static_assert(kCompactIters * kFmtWaves <= kWave, "one wavefront scans the tile's per-wave counts");
  if (wave == 0) {   // exclusive prefix of the (iteration, wave) counts, in the order the edges are numbered
    const uint32_t c = lane < kCompactIters * kFmtWaves ? s_cnt[lane] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < kCompactIters * kFmtWaves; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    if (lane < kCompactIters * kFmtWaves) s_cnt[lane] = first + incl - c;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kCompactIters; ++it) {
    const int64_t s = base + it * kFmtBlock + threadIdx.x;
    if (s >= upper) continue;
    const int64_t e = static_cast<int64_t>(s_cnt[it * kFmtWaves + wave]) + below[it];
    // (slot numbers fit 32 bits, fmt_sizes_ok: a 32-bit division, a fraction of the cost of a 64-bit one)
    const uint32_t fan = static_cast<uint32_t>(p.fanout);
    const uint32_t d = static_cast<uint32_t>(s) / fan;
    // Valid slots before the first slot of a destination = its CSC offset;
    // destinations past the device-side count get the edge total (empty rows).
    if (static_cast<uint32_t>(s) - d * fan == 0) p.csc_indptr[d] = e;
    if (v[it] >= 0) {
      p.coo_row[e] = v[it];
      p.coo_col[e] = d;
    }
  }
}

// ------------------------------------------------------------------- CSR
struct SortParams {
  const int64_t* coo_row;     // keys of the first pass
  const int64_t* coo_col;
  const int64_t* num_edges_dev;
  int64_t max_edges;
  const uint32_t* key_in;     // later passes
  const uint32_t* pay_in;
  uint32_t* key_out;
  uint32_t* pay_out;
  // fused: [tiles][kRadix] counts; else [kRadix][tiles], each digit's row scanned over tiles
  uint32_t* tile_hist;
  uint32_t* bin_total;        // [kRadix] (not fused)
  int64_t tiles;
  bool fused;
  int shift;
  int64_t* csr_indices;       // last pass
  int64_t* csr_eids;
};

template <bool FIRST>
__device__ __forceinline__ uint32_t sort_key(const SortParams& p, int64_t i) {
  return FIRST ? static_cast<uint32_t>(p.coo_row[i]) : p.key_in[i];
}

template <bool FIRST>
__global__ __launch_bounds__(kSortBlock) void radix_hist_kernel(SortParams p) {
  __shared__ uint32_t s_hist[kRadix];
  const int tid = threadIdx.x;
  s_hist[tid] = 0;
  __syncthreads();
  const int64_t n = actual_count(p.max_edges, p.num_edges_dev);
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSortTile;
  // all of a thread's keys are requested before the first is counted
  uint32_t key[kSortTile / kSortBlock];
#pragma unroll
  for (int k = 0; k < kSortTile / kSortBlock; ++k) {
    const int64_t i = base + k * kSortBlock + tid;
    key[k] = i < n ? sort_key<FIRST>(p, i) : 0u;
  }
#pragma unroll
  for (int k = 0; k < kSortTile / kSortBlock; ++k)
    if (base + k * kSortBlock + tid < n) atomicAdd(&s_hist[(key[k] >> p.shift) & (kRadix - 1)], 1u);
  __syncthreads();
  const int64_t at = p.fused ? static_cast<int64_t>(blockIdx.x) * kRadix + tid
                             : static_cast<int64_t>(tid) * p.tiles + blockIdx.x;
  p.tile_hist[at] = s_hist[tid];
}

// One workgroup per digit: exclusive prefix of its row of tile_hist over the tiles.
__global__ __launch_bounds__(kSortBlock) void radix_binscan_kernel(SortParams p) {
  __shared__ uint32_t s_wave[kSortWaves];
  uint32_t* row = p.tile_hist + static_cast<int64_t>(blockIdx.x) * p.tiles;
  const int64_t n = actual_count(p.max_edges, p.num_edges_dev);
  const int64_t active = ceil_div_dev(n, kSortTile);
  uint32_t carry = 0;
  for (int64_t c0 = 0; c0 < active; c0 += kSortBlock) {
    const int64_t i = c0 + threadIdx.x;
    const uint32_t x = i < active ? row[i] : 0u;
    uint32_t all;
    const uint32_t excl = block_exclusive(x, s_wave, all);
    if (i < active) row[i] = carry + excl;
    carry += all;
  }
  if (threadIdx.x == 0) p.bin_total[blockIdx.x] = carry;
}

template <bool FIRST, bool LAST>
__global__ __launch_bounds__(kSortBlock) void radix_scatter_kernel(SortParams p) {
  // s_pos[w][b]: next position, inside the tile's digit-sorted order, of digit b
  // for wave w.  A wave owns kSortWaveItems consecutive items, so walking waves
  // in order, and rounds in order inside a wave, keeps equal digits in input
  // order.  Items are first put into that order in LDS and then written out, so
  // that neighbouring lanes write neighbouring addresses (a digit's run).
  __shared__ uint32_t s_pos[kSortWaves][kRadix];
  __shared__ uint32_t s_delta[kRadix];     // output position = s_delta[digit] + position in the tile's order
  __shared__ uint32_t s_wave[kSortWaves];
  __shared__ uint32_t s_key[kSortTile];
  __shared__ uint32_t s_pay[kSortTile];
  const int tid = threadIdx.x;             // = digit in the per-digit steps
  const int lane = lane_id();
  const int wave = tid / kWave;
  const int64_t n = actual_count(p.max_edges, p.num_edges_dev);
  const int64_t tile_base = static_cast<int64_t>(blockIdx.x) * kSortTile;
  if (tile_base >= n) return;  // block-uniform
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) s_pos[w][tid] = 0;
  __syncthreads();
  const int64_t wave_base = tile_base + static_cast<int64_t>(wave) * kSortWaveItems;
  uint32_t key[kSortRounds], pay[kSortRounds];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {   // every load of the lane is requested before the first is used
    const int64_t i = wave_base + r * kWave + lane;
    key[r] = i < n ? sort_key<FIRST>(p, i) : 0u;
    pay[r] = FIRST ? static_cast<uint32_t>(i) : (i < n ? p.pay_in[i] : 0u);
  }
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
    if (wave_base + r * kWave + lane < n) atomicAdd(&s_pos[wave][(key[r] >> p.shift) & (kRadix - 1)], 1u);
  // First output position of this tile's items of digit `tid`: items with a
  // smaller digit anywhere, plus items with the same digit in earlier tiles.
  uint32_t first;
  if (p.fused) {
    const int64_t active = ceil_div_dev(n, kSortTile);
    uint32_t before = 0, total = 0;
    for (int64_t t0 = 0; t0 < active; t0 += 8) {
      uint32_t c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] = t0 + u < active ? p.tile_hist[(t0 + u) * kRadix + tid] : 0u;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        total += c[u];
        if (t0 + u < blockIdx.x) before += c[u];
      }
    }
    uint32_t all;
    first = block_exclusive(total, s_wave, all) + before;
  } else {
    // tile_hist[digit][tile] already holds the prefix over tiles; bin_total the digit's count
    uint32_t all;
    first = block_exclusive(p.bin_total[tid], s_wave, all) +
            p.tile_hist[static_cast<int64_t>(tid) * p.tiles + blockIdx.x];
  }
  __syncthreads();
  uint32_t mine_total = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) mine_total += s_pos[w][tid];
  uint32_t all;
  uint32_t local = block_exclusive(mine_total, s_wave, all);   // digit's start inside the tile
  s_delta[tid] = first - local;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    const uint32_t c = s_pos[w][tid];
    s_pos[w][tid] = local;
    local += c;
  }
  __syncthreads();
  volatile uint32_t* mine = s_pos[wave];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const int64_t i = wave_base + r * kWave + lane;
    const bool valid = i < n;
    const uint32_t d = valid ? (key[r] >> p.shift) & (kRadix - 1) : 0u;
    uint64_t peers = ballot(valid);
#pragma unroll
    for (int b = 0; b < kRadixBits; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t set = ballot(valid && bit);
      peers &= bit ? set : ~set;
    }
    const uint32_t rank = rank_below(peers);
    uint32_t pos = 0;
    if (valid) pos = mine[d] + rank;
    __builtin_amdgcn_wave_barrier();
    // the last lane of a digit's group moves the counter past the group
    if (valid && rank + 1 == static_cast<uint32_t>(__popcll(peers))) mine[d] = pos + 1;
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      s_key[pos] = key[r];
      s_pay[pos] = pay[r];
    }
  }
  __syncthreads();
  const int count = static_cast<int>(min(static_cast<int64_t>(kSortTile), n - tile_base));
  // (in the last pass an item's destination is a dependent read: all of a thread's are requested before any store)
  int64_t col[LAST ? kSortRounds : 1];
  if (LAST) {
#pragma unroll
    for (int q = 0; q < kSortRounds; ++q) {
      const int j = q * kSortBlock + tid;
      col[q] = j < count ? p.coo_col[s_pay[j]] : 0;
    }
  }
#pragma unroll
  for (int q = 0; q < kSortRounds; ++q) {
    const int j = q * kSortBlock + tid;
    if (j >= count) break;
    const uint32_t k = s_key[j];
    const uint32_t v = s_pay[j];
    const uint32_t pos = s_delta[(k >> p.shift) & (kRadix - 1)] + j;
    if (LAST) {
      p.csr_eids[pos] = v;
      p.csr_indices[pos] = col[q];
    } else {
      p.pay_out[pos] = v;
    }
    p.key_out[pos] = k;
  }
}

// ---------------------------------------------------- CSR by source ranges
// Sources are cut into ranges.  The compaction's count pass also counts a tile's
// edges per range, one launch turns the counts into prefixes over the tiles, the
// place pass (which knows an edge's id, source and destination) puts a packed
// record of every edge into its range's part of a scratch array, in edge order, and
// one workgroup per range sorts its records by source in LDS and writes offsets,
// destinations and edge ids.  Two stable passes instead of three to four, and none
// of them over a few tiles only (a radix pass over the 260 k edges of a batch of
// 1024 is 64 workgroups on 256 CUs).  All three formats of a block, with radix
// passes / with ranges, sizes exact: 8 k edges 40 / 22 us, 22 k 41 / 25, 260 k
// (120 k sources) 79 / 33, 740 k (240 k) 88 / 49, 940 k (460 k) 89 / 50 us.  With edges in long ranges (1 M edges; one
// source in every tenth slot, with a low / a high id): 98 / 55, 98 / 73; all edges in one: 96 / 64, 294 / 132; four
// sources in four of ten slots: 97 / 86 us.
// The relabel numbers nodes by first occurrence, so hubs have small ids and the
// edges per source fall off about as 1 / id (2.4 M-node graph, 4096 seeds: 40 edges
// per source at id 4500, 5 at 30 k, 1.4 at 200 k), and buffers sized by upper bounds
// end in ids that do not occur.  Ranges of equal width would leave one workgroup with
// 37 k records (93 us); four widths keep them between a few hundred and a few thousand.
constexpr int kRangeMaxShift = 11;
// The first sources have a range each: the worst hubs, and all sources of a block that has few.  Such a range needs no
// sort, so any number of workgroups may share it (range_sort_kernel).
constexpr int64_t kRangeFrom0 = 256;                                                // sources with a range each
constexpr int64_t kRangeFrom1 = int64_t{1} << 15, kRangeFrom2 = int64_t{1} << 18;   // first sources of pieces 1, 2
constexpr int kRangeShift0 = 5, kRangeShift1 = 8, kRangeShift2 = 10;
constexpr int kRangeMaxCount = 5016;          // ranges: 12 bytes of LDS each in the place pass
constexpr int64_t kRangeMaxTiles = 4096;
// A tile of the partition: 1024 slots (four per thread) instead of 2048 while the edges are few and workgroups with them.
// Every tile walks all ranges, so a large block is better off with half the tiles.  CSR of 8 k / 260 k / 730 k / 950 k /
// 3.4 M edges with 2048 and 1024: 51 / 47, 114 / 108, 183 / 191, 198 / 210, 476 / 542 us (host reads included).
// A row count in device memory is usually a fraction of its bound (a batch of the 111 M-node graph: 1.07 M edges for bounds
// of 4.3 M slots), so the bound may be four times that; a block that fills it pays the 6 to 8 % above.
constexpr int64_t kRangeSmallSlots = int64_t{1} << 19, kRangeSmallBound = int64_t{1} << 21;
constexpr int kRangeSmallIters = 4;
constexpr int kRangeKeyBits = kRangeMaxShift;
constexpr int kRangeEdgeBits = 32;
constexpr int64_t kRangeMaxDst = int64_t{1} << (64 - kRangeKeyBits - kRangeEdgeBits);
constexpr int kRangeSortBlock = 256;
constexpr int kRangeSortWaves = kRangeSortBlock / kWave;
constexpr int kRangeSortRounds = 8;
constexpr int kRangeSortChunk = kRangeSortBlock * kRangeSortRounds;
// A range of more records than four times the mean is sorted in parts, within these bounds.
constexpr int64_t kRangeLong = 2 * kRangeSortChunk, kRangeLongest = 8 * kRangeSortChunk;
constexpr int kRangePart = kRangeSortChunk;            // records of a part: this many, or a 64th of the range
constexpr int kRangeMaxParts = 64;
constexpr int kRangePartGroups = 512;
constexpr int kRangeScanGroups = 16;          // tile groups of a scan workgroup

struct RangeParams {
  int shift2;                 // width of piece 2
  int ranges;
  int tile;                   // slots of a workgroup
  int part_groups;            // workgroups of the sort that take parts of long ranges
  uint32_t long_from;         // a range of more records is sorted in parts
  int row_words;              // keys of the widest range
  uint32_t* parts;            // [1]: number of parts
  uint32_t* part0;            // [ranges]: a long range's first part
  uint32_t* part_range;       // [parts]
  uint32_t* part_keys;        // [parts][row_words]: records of a part per source
  uint32_t* hist;             // [tiles][ranges]: edges of a tile per range, then their prefix over the tiles
  uint32_t* total;            // [ranges]
  uint32_t* start;            // [ranges + 1]: a range's first record
  uint64_t* rec;              // edges by range: destination | source within the range | edge id
  int64_t num_src;
  int64_t* csr_indptr;
  int64_t* csr_indices;
  int64_t* csr_eids;
  uint32_t* t_indptr;         // transpose only (apt_block_transpose)
  uint32_t* t_slots;
  LongRows lng;               // sources with very many edges: the table that the sums over them read
};

constexpr int kRangeSingles = static_cast<int>(kRangeFrom0);
constexpr int kRangeCount0 = kRangeSingles + static_cast<int>((kRangeFrom1 - kRangeFrom0) >> kRangeShift0);   // ranges up to piece 1
constexpr int kRangeCount1 = static_cast<int>((kRangeFrom2 - kRangeFrom1) >> kRangeShift1);

__host__ __device__ __forceinline__ int64_t range_index(int64_t src, int shift2) {
  return src < kRangeFrom0   ? src
         : src < kRangeFrom1 ? kRangeSingles + ((src - kRangeFrom0) >> kRangeShift0)
         : src < kRangeFrom2 ? kRangeCount0 + ((src - kRangeFrom1) >> kRangeShift1)
                             : kRangeCount0 + kRangeCount1 + ((src - kRangeFrom2) >> shift2);
}
__device__ __forceinline__ int range_shift(const RangeParams& r, int b) {
  return b < kRangeSingles ? 0 : b < kRangeCount0 ? kRangeShift0 : b < kRangeCount0 + kRangeCount1 ? kRangeShift1 : r.shift2;
}
__device__ __forceinline__ int64_t range_first(const RangeParams& r, int b) {
  return b < kRangeSingles ? b
         : b < kRangeCount0 ? kRangeFrom0 + (static_cast<int64_t>(b - kRangeSingles) << kRangeShift0)
         : b < kRangeCount0 + kRangeCount1 ? kRangeFrom1 + (static_cast<int64_t>(b - kRangeCount0) << kRangeShift1)
                                           : kRangeFrom2 + (static_cast<int64_t>(b - kRangeCount0 - kRangeCount1) << r.shift2);
}
// Sources past num_src (they have no offset of their own) sort behind those that have one, in the last range.
__device__ __forceinline__ int range_of(const RangeParams& r, int64_t src) {
  const int64_t b = range_index(src, r.shift2);
  return b < r.ranges ? static_cast<int>(b) : r.ranges - 1;
}
__device__ __forceinline__ uint32_t range_key(const RangeParams& r, int b, int64_t src) {
  const int64_t k = src - range_first(r, b), last = (int64_t{1} << range_shift(r, b)) - 1;
  return static_cast<uint32_t>(k < last ? k : last);
}

__device__ __forceinline__ uint32_t part_length(uint32_t n) {   // a multiple of a chunk
  return max(static_cast<uint32_t>(kRangePart), (n / kRangeMaxParts + kRangeSortChunk) / kRangeSortChunk * kRangeSortChunk);
}
__device__ __forceinline__ uint32_t part_count(uint32_t n) { return (n + part_length(n) - 1) / part_length(n); }

// Lanes of the wavefront that hold the same value (its low `bits` bits) as this one, among `valid` lanes.
__device__ __forceinline__ uint64_t same_value(uint32_t v, int bits, bool valid) {
  uint64_t peers = ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (v >> b) & 1u;
    const uint64_t set = ballot(valid && bit);
    peers &= bit ? set : ~set;
  }
  return peers;
}

// FORMATS: COO, CSC and CSR (an edge's id is its place in the COO).  Otherwise the transpose alone: the edges of a
// source by slot, without a compaction.
template <bool FORMATS, int ITERS>
__global__ __launch_bounds__(kFmtBlock) void range_count_kernel(CompactParams p, RangeParams r) {
  extern __shared__ uint32_t s_range[];   // [ranges]
  __shared__ uint32_t s_wave[kFmtWaves];
  const int64_t slots = actual_count(p.num_dst, p.num_dst_dev) * p.fanout;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kFmtBlock * ITERS);
  if (base >= slots && blockIdx.x != 0) return;   // block-uniform: nobody reads an inactive tile's counts
  if (blockIdx.x == 0 && threadIdx.x == 0) *r.parts = 0;
  if (!FORMATS)
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kFmtBlock + threadIdx.x; i < r.lng.slots;
         i += static_cast<int64_t>(gridDim.x) * kFmtBlock)
      r.lng.row[i] = r.lng.arrived[i] = 0;
  int64_t v[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int64_t s = base + it * kFmtBlock + threadIdx.x;
    v[it] = s < slots ? p.relabeled[s] : -1;
  }
  for (int b = threadIdx.x; b < r.ranges; b += kFmtBlock) s_range[b] = 0;
  __syncthreads();
  uint32_t c = 0;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    if (v[it] < 0) continue;
    ++c;
    atomicAdd(&s_range[range_of(r, v[it])], 1u);
  }
  if (FORMATS) {
    uint32_t all;
    block_exclusive(c, s_wave, all);
    if (threadIdx.x == 0) p.tile_cnt[blockIdx.x] = all;
  }
  __syncthreads();
  uint32_t* row = r.hist + static_cast<int64_t>(blockIdx.x) * r.ranges;
  for (int b = threadIdx.x; b < r.ranges; b += kFmtBlock) row[b] = s_range[b];
}

// 64 ranges per workgroup, the tiles in kRangeScanGroups groups: a group adds up its tiles, the groups' sums are
// put in order in LDS, and a second walk leaves the prefixes.
__global__ __launch_bounds__(kWave * kRangeScanGroups) void range_scan_kernel(CompactParams p, RangeParams r) {
  constexpr int kUnroll = 8;
  __shared__ uint32_t s_sum[kRangeScanGroups][kWave];
  __shared__ uint32_t s_part0[kWave];
  const int lane = threadIdx.x % kWave, group = threadIdx.x / kWave;
  const int b = blockIdx.x * kWave + lane;
  const int64_t slots = actual_count(p.num_dst, p.num_dst_dev) * p.fanout;
  const int tiles = static_cast<int>(ceil_div_dev(slots, r.tile));
  const int per = (tiles + kRangeScanGroups - 1) / kRangeScanGroups;
  const int t0 = group * per, t1 = min(t0 + per, tiles);
  const bool live = b < r.ranges;
  uint32_t sum = 0;
  for (int t = t0; t < t1 && live; t += kUnroll) {
    uint32_t c[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) c[u] = r.hist[static_cast<int64_t>(min(t + u, t1 - 1)) * r.ranges + b];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) sum += t + u < t1 ? c[u] : 0u;
  }
  s_sum[group][lane] = sum;
  __syncthreads();
  uint32_t run = 0, all = 0;
#pragma unroll
  for (int g = 0; g < kRangeScanGroups; ++g) {
    const uint32_t c = s_sum[g][lane];
    if (g < group) run += c;
    all += c;
  }
  uint64_t lengthy = ballot(live && all > r.long_from);   // (every wavefront has the same lanes' totals)
  if (lengthy != 0) {   // block-uniform: number their parts, and clear the counts that the place pass adds to
    if (group == 0 && ((lengthy >> lane) & 1)) {
      const uint32_t parts = part_count(all), part0 = atomicAdd(r.parts, parts);
      r.part0[b] = s_part0[lane] = part0;
      for (uint32_t q = 0; q < parts; ++q) r.part_range[part0 + q] = b;
    }
    __syncthreads();
    for (; lengthy != 0; lengthy &= lengthy - 1) {
      const int src = __ffsll(static_cast<long long>(lengthy)) - 1;
      const int keys = 1 << range_shift(r, blockIdx.x * kWave + src);
      const uint32_t words = keys > 1 ? part_count(__shfl(all, src, kWave)) * r.row_words : 0u;
      uint32_t* row = r.part_keys + static_cast<int64_t>(s_part0[src]) * r.row_words;
      for (uint32_t i = threadIdx.x; i < words; i += kWave * kRangeScanGroups) row[i] = 0;
    }
  }
  if (!live) return;
  for (int t = t0; t < t1; t += kUnroll) {
    uint32_t c[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) c[u] = r.hist[static_cast<int64_t>(min(t + u, t1 - 1)) * r.ranges + b];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      if (t + u < t1) {
        r.hist[static_cast<int64_t>(t + u) * r.ranges + b] = run;
        run += c[u];
      }
  }
  if (group == 0) r.total[b] = all;
}

// The compaction's place pass (as fmt_place_kernel) with the partition: a wavefront owns consecutive slots, so that
// walking the wavefronts, and the iterations inside one, is edge order.
template <bool FORMATS, int ITERS>
__global__ __launch_bounds__(kFmtBlock) void range_place_kernel(CompactParams p, RangeParams r) {
  extern __shared__ uint32_t s_range[];
  uint32_t* s_base = s_range;                                                // [ranges]
  uint32_t* s_cnt2 = s_range + r.ranges;                                     // [waves][ranges / 2], 16-bit counts
  const int words = (r.ranges + 1) / 2;                                      // 32-bit words of a wave's counts
  __shared__ uint32_t s_edges[kFmtWaves * ITERS];
  __shared__ uint32_t s_wave[kFmtWaves];
  __shared__ int s_long;                                                     // whether there are long ranges
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const int64_t slots = actual_count(p.num_dst, p.num_dst_dev) * p.fanout;
  const int64_t upper = p.num_dst * p.fanout;
  if (threadIdx.x == 0) s_long = 0;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kFmtBlock * ITERS) + wave * (ITERS * kWave);
  int64_t v[ITERS];
  uint32_t below[ITERS];
  int range[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int64_t s = base + it * kWave + lane;
    v[it] = s < slots ? p.relabeled[s] : -1;
  }
  for (int i = threadIdx.x; i < words * kFmtWaves; i += kFmtBlock) s_cnt2[i] = 0;
  __syncthreads();
  uint32_t* cnt = s_cnt2 + wave * words;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const uint64_t m = ballot(v[it] >= 0);
    below[it] = rank_below(m);
    if (lane == 0) s_edges[wave * ITERS + it] = __popcll(m);
    range[it] = v[it] >= 0 ? range_of(r, v[it]) : 0;
    if (v[it] >= 0)   // at most 512 per wavefront: a 16-bit half never overflows into the other
      atomicAdd(&cnt[range[it] >> 1], (range[it] & 1) ? 0x10000u : 1u);
  }
  const int64_t active = ceil_div_dev(slots, (kFmtBlock * ITERS));
  uint32_t first = 0;
  if (FORMATS) {   // edges of the tiles before this one, and of all tiles
    uint32_t before = 0, total = 0, all_total;
    for (int64_t t = threadIdx.x; t < active; t += kFmtBlock) {
      const uint32_t c = p.tile_cnt[t];
      total += c;
      if (t < blockIdx.x) before += c;
    }
    block_exclusive(before, s_wave, first);
    block_exclusive(total, s_wave, all_total);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *p.num_edges_dev = all_total;
      p.csc_indptr[p.num_dst] = all_total;
    }
  } else {
    __syncthreads();   // the counts are complete
  }
  // where this tile's edges of a range start: the ranges before it, and the tiles before this one
  const bool live = blockIdx.x < active || blockIdx.x == 0;   // block-uniform (workgroup 0 also writes the starts)
  if (live) {
    // (loads of a thread in batches: one at a time, a workgroup of a large launch would spend its time on them)
    constexpr int kBatch = 6;
    for (int b = threadIdx.x; b < r.ranges; b += kBatch * kFmtBlock) {
      uint32_t c[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) c[u] = r.total[min(b + u * kFmtBlock, r.ranges - 1)];
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (b + u * kFmtBlock < r.ranges) {
          s_base[b + u * kFmtBlock] = c[u];
          if (c[u] > r.long_from && b + u * kFmtBlock >= kRangeSingles) s_long = 1;
        }
    }
    __syncthreads();
    const int per = (r.ranges + kFmtBlock - 1) / kFmtBlock;
    const int b0 = threadIdx.x * per, b1 = min(b0 + per, r.ranges);
    uint32_t mine = 0;
    for (int b = b0; b < b1; ++b) mine += s_base[b];
    uint32_t all;
    uint32_t run = block_exclusive(mine, s_wave, all);
    for (int b = b0; b < b1; ++b) {
      const uint32_t c = s_base[b];
      s_base[b] = run;
      run += c;
    }
    __syncthreads();
    const uint32_t* row = r.hist + static_cast<int64_t>(blockIdx.x) * r.ranges;
    for (int b = threadIdx.x; b < r.ranges; b += kBatch * kFmtBlock) {
      uint32_t c[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) c[u] = row[min(b + u * kFmtBlock, r.ranges - 1)];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = b + u * kFmtBlock;
        if (i >= r.ranges) break;
        if (blockIdx.x == 0) r.start[i] = s_base[i];
        s_base[i] += c[u];
      }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) r.start[r.ranges] = all;
    // counts of a wavefront -> counts of the wavefronts before it
    for (int i = threadIdx.x; i < words; i += kFmtBlock) {
      uint32_t sum = 0;
#pragma unroll
      for (int w = 0; w < kFmtWaves; ++w) {
        const uint32_t c = s_cnt2[w * words + i];
        s_cnt2[w * words + i] = sum;
        sum += c;
      }
    }
  }
  static_assert(ITERS * kFmtWaves <= kWave, "one wavefront scans the tile's per-wave counts");
  if (FORMATS && wave == 0) {
    const uint32_t c = lane < ITERS * kFmtWaves ? s_edges[lane] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < ITERS * kFmtWaves; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    if (lane < ITERS * kFmtWaves) s_edges[lane] = first + incl - c;
  }
  __syncthreads();
  const int bits = 32 - __clz(r.ranges - 1 > 0 ? r.ranges - 1 : 1);
  volatile uint16_t* pos = reinterpret_cast<volatile uint16_t*>(cnt);
  const uint32_t fan = static_cast<uint32_t>(p.fanout);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int64_t s = base + it * kWave + lane;
    const int64_t e = FORMATS ? static_cast<int64_t>(s_edges[wave * ITERS + it]) + below[it] : s;
    const uint32_t d = FORMATS ? static_cast<uint32_t>(s) / fan : 0u;
    if (FORMATS && s < upper && static_cast<uint32_t>(s) - d * fan == 0) p.csc_indptr[d] = e;
    const bool valid = v[it] >= 0;
    if (ballot(valid) == 0) continue;   // wave-uniform
    const uint32_t b = static_cast<uint32_t>(range[it]);
    const uint64_t peers = same_value(b, bits, valid);
    const uint32_t rank = rank_below(peers);
    uint32_t at = 0;
    if (valid) at = pos[b] + rank;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank + 1 == static_cast<uint32_t>(__popcll(peers))) pos[b] = static_cast<uint16_t>(at + 1);
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      if (FORMATS) {
        p.coo_row[e] = v[it];
        p.coo_col[e] = d;
      }
      r.rec[s_base[b] + at] = (static_cast<uint64_t>(d) << (kRangeKeyBits + kRangeEdgeBits)) |
                              (static_cast<uint64_t>(range_key(r, static_cast<int>(b), v[it])) << kRangeEdgeBits) | static_cast<uint64_t>(e);
    }
    if (s_long != 0) {   // block-uniform: count the edges of a long range's part per source
      const uint32_t n = r.total[b];
      const bool count = valid && b >= static_cast<uint32_t>(kRangeSingles) && n > r.long_from;
      uint32_t cell = 0;
      if (count) {
        const uint32_t before = r.hist[static_cast<int64_t>(blockIdx.x) * r.ranges + b] + at;   // records of the range
        cell = (r.part0[b] + before / part_length(n)) * r.row_words + range_key(r, static_cast<int>(b), v[it]);
      }
      uint64_t todo = ballot(count);
      for (int t = 0; t < 4 && todo != 0; ++t) {   // a hub's lanes together, the others by themselves
        const int leader = __ffsll(static_cast<long long>(todo)) - 1;
        const uint64_t same = ballot(cell == __shfl(cell, leader, kWave)) & todo;
        if (lane == leader) atomicAdd(&r.part_keys[cell], static_cast<uint32_t>(__popcll(same)));
        todo &= ~same;
      }
      if ((todo >> lane) & 1) atomicAdd(&r.part_keys[cell], 1u);
    }
  }
}

// One workgroup per range: stable counting sort of its records by source.  A range of a sampled block has about a
// thousand; one with more than a chunk of them is walked chunk by chunk, after a counting walk.  A long range (a hub, or
// a block of few sources) would keep its workgroup busy long after the others are done: it is cut into parts for the
// first `part_groups` workgroups of the launch.  The place pass has counted a long range's records per part and source.
template <bool FORMATS>
__global__ __launch_bounds__(kRangeSortBlock) void range_sort_kernel(RangeParams r) {
  extern __shared__ uint32_t s_range[];
  __shared__ uint32_t s_wave[kRangeSortWaves];
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  auto exclusive = [&](uint32_t x, uint32_t& all) {   // over the workgroup
    uint32_t incl = x;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    __syncthreads();
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    all = 0;
#pragma unroll
    for (int w = 0; w < kRangeSortWaves; ++w) {
      const uint32_t c = s_wave[w];
      if (w < wave) before += c;
      all += c;
    }
    return before + incl - x;
  };
  // Records [first, last) of range b (of which it has n, from position `before` on); part0: the range's first part if
  // it is long.
  auto sort = [&](int b, uint32_t before, uint32_t n, uint32_t first, uint32_t last, bool part, uint32_t part0) {
    const int shift = range_shift(r, b);
    const int keys = 1 << shift;
    const int words = keys / 2;
    uint32_t* s_start = s_range;              // [keys]: next position of a key's first record not yet placed
    uint32_t* s_cnt2 = s_range + keys;        // [waves][keys / 2], 16-bit counts
    uint32_t* s_before = s_cnt2;              // [keys], before those: records ahead of `first`
    const int64_t src0 = range_first(r, b);
    auto set_offset = [&](int k, uint32_t at, uint32_t count) {
      if (src0 + k > r.num_src) return;
      if (FORMATS) {
        r.csr_indptr[src0 + k] = at;
      } else {
        r.t_indptr[src0 + k] = at;
        if (r.lng.slots > 0 && count > r.lng.longer && src0 + k < r.num_src)
          r.lng.row[at / r.lng.longer] = static_cast<uint32_t>(src0 + k) + 1;
      }
    };
    if (n == 0) {
      for (int k = tid; k < keys; k += kRangeSortBlock) set_offset(k, before, 0);
      return;
    }
    const uint64_t* rec = r.rec + before;
    auto place = [&](int64_t to, uint64_t x) {
      const uint32_t e = static_cast<uint32_t>(x);
      if (FORMATS) {
        r.csr_eids[to] = e;
        r.csr_indices[to] = static_cast<int64_t>(x >> (kRangeKeyBits + kRangeEdgeBits));
      } else {
        r.t_slots[to] = e;
      }
    };
    if (keys == 1) {   // one source: its records are in order already
      if (first == 0 && tid == 0) set_offset(0, before, n);
      for (uint32_t i = first + tid; i < last; i += kRangeSortBlock) place(static_cast<int64_t>(before) + i, rec[i]);
      return;
    }
    auto key_of = [&](uint64_t x) { return static_cast<uint32_t>(x >> kRangeEdgeBits) & ((1u << kRangeKeyBits) - 1); };
    const bool single = n <= kRangeSortChunk;   // block-uniform
    const int per = (keys + kRangeSortBlock - 1) / kRangeSortBlock;
    // counts per key in s_start -> the key's first position, and its offset
    auto starts = [&]() {
      const int k0 = tid * per, k1 = min(k0 + per, keys);
      uint32_t mine = 0, all;
      for (int k = k0; k < k1; ++k) mine += s_start[k];
      uint32_t run = exclusive(mine, all);
      for (int k = k0; k < k1; ++k) {
        const uint32_t c = s_start[k];
        s_start[k] = run;
        if (first == 0) set_offset(k, before + run, c);
        run += c;
      }
    };
    if (part) {
      constexpr int kBatch = 8;
      const uint32_t parts = part_count(n), mine = first / part_length(n);
      for (int k = tid; k < keys; k += kRangeSortBlock) {
        const uint32_t* col = r.part_keys + static_cast<int64_t>(part0) * r.row_words + k;
        uint32_t total = 0, ahead = 0;
        for (uint32_t q = 0; q < parts; q += kBatch) {
          uint32_t c[kBatch];
#pragma unroll
          for (int u = 0; u < kBatch; ++u) c[u] = col[static_cast<int64_t>(min(q + u, parts - 1)) * r.row_words];
#pragma unroll
          for (int u = 0; u < kBatch; ++u) {
            total += q + u < parts ? c[u] : 0u;
            ahead += q + u < mine ? c[u] : 0u;
          }
        }
        s_start[k] = total;
        s_before[k] = ahead;
      }
      __syncthreads();
      starts();
      __syncthreads();
      for (int k = tid; k < keys; k += kRangeSortBlock) s_start[k] += s_before[k];
    } else if (!single) {
      for (int k = tid; k < keys; k += kRangeSortBlock) s_start[k] = 0;
      __syncthreads();
      for (uint32_t i = tid; i < n; i += kRangeSortBlock) atomicAdd(&s_start[key_of(rec[i])], 1u);
      __syncthreads();
      starts();
    }
    uint32_t* cnt = s_cnt2 + wave * words;
    volatile uint16_t* pos = reinterpret_cast<volatile uint16_t*>(cnt);
    for (uint32_t c0 = first; c0 < last; c0 += kRangeSortChunk) {
      const uint32_t left = min(last - c0, static_cast<uint32_t>(kRangeSortChunk));
      const int rounds = static_cast<int>((left + kRangeSortBlock - 1) / kRangeSortBlock);
      uint64_t x[kRangeSortRounds];
#pragma unroll
      for (int q = 0; q < kRangeSortRounds; ++q) {
        const uint32_t i = (wave * rounds + q) * kWave + lane;
        x[q] = q < rounds && i < left ? rec[c0 + i] : ~0ull;
      }
      __syncthreads();
      for (int i = tid; i < words * kRangeSortWaves; i += kRangeSortBlock) s_cnt2[i] = 0;
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kRangeSortRounds; ++q)
        if (x[q] != ~0ull) {
          const uint32_t k = key_of(x[q]);
          atomicAdd(&cnt[k >> 1], (k & 1) ? 0x10000u : 1u);
        }
      __syncthreads();
      // counts of a wavefront -> counts of the wavefronts before it (a chunk's 2048 fit 16 bits)
      for (int i = tid; i < words; i += kRangeSortBlock) {
        uint32_t sum = 0;
#pragma unroll
        for (int w = 0; w < kRangeSortWaves; ++w) {
          const uint32_t c = s_cnt2[w * words + i];
          s_cnt2[w * words + i] = sum;
          sum += c;
        }
        if (single) {
          s_start[2 * i] = sum & 0xffffu;
          s_start[2 * i + 1] = sum >> 16;
        }
      }
      __syncthreads();
      if (single) {
        starts();
        __syncthreads();
      }
#pragma unroll
      for (int q = 0; q < kRangeSortRounds; ++q) {
        if (q >= rounds) break;   // block-uniform
        const bool valid = x[q] != ~0ull;
        const uint32_t k = valid ? key_of(x[q]) : 0u;
        const uint64_t peers = same_value(k, shift, valid);
        const uint32_t rank = rank_below(peers);
        uint32_t at = 0;
        if (valid) at = pos[k] + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank + 1 == static_cast<uint32_t>(__popcll(peers))) pos[k] = static_cast<uint16_t>(at + 1);
        __builtin_amdgcn_wave_barrier();
        if (valid) place(static_cast<int64_t>(before) + s_start[k] + at, x[q]);
      }
      if (c0 + kRangeSortChunk >= last) break;
      __syncthreads();
      // every wavefront has moved its counters past its records: the last one's stand at the chunk's totals
      const uint16_t* moved = reinterpret_cast<const uint16_t*>(s_cnt2 + (kRangeSortWaves - 1) * words);
      for (int k = tid; k < keys; k += kRangeSortBlock) s_start[k] += moved[k];
    }
  };
  const bool whole = static_cast<int>(blockIdx.x) >= r.part_groups;   // a range of its own
  const uint32_t parts = whole ? 0u : *r.parts;
  for (uint32_t p = blockIdx.x;; p += r.part_groups) {   // block-uniform
    if (!whole && p >= parts) return;
    const int b = whole ? static_cast<int>(blockIdx.x) - r.part_groups : static_cast<int>(r.part_range[p]);
    const uint32_t before = r.start[b], n = r.start[b + 1] - before;
    const bool part = n > r.long_from;
    if (whole && part) return;
    const uint32_t part0 = whole ? 0u : r.part0[b], first = whole ? 0u : (p - part0) * part_length(n);
    sort(b, before, n, first, whole ? n : min(first + part_length(n), n), part, part0);
    if (whole) return;
    __syncthreads();   // (the counters)
  }
}

// csr_indptr[s] = first position of a key >= s in the sorted keys, s in [0, num_src].
// Position e starts a run of its key k when the key before it, kp, is smaller: then e is the answer for every
// s in (kp, k].  One lane per position writes those entries itself when they are few (in a sampled block nearly
// every source has an edge, so the run before a key is one or two entries long); a longer stretch is filled by the
// whole wavefront.  Sources above the largest key get the edge total.  No searching: every offset is written
// once, from a coalesced read of the keys.
constexpr int kIndptrShortGap = 4;

__global__ __launch_bounds__(kFmtBlock) void csr_indptr_kernel(const uint32_t* __restrict__ keys,
                                                               const int64_t* num_edges_dev, int64_t max_edges,
                                                               int64_t num_src, int64_t* __restrict__ csr_indptr) {
  const int64_t n = actual_count(max_edges, num_edges_dev);
  const int64_t last = n > 0 ? static_cast<int64_t>(keys[n - 1]) : -1;
  const int lane = lane_id();
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * kFmtBlock + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kFmtBlock;
  for (int64_t e0 = tid - lane; e0 < n; e0 += stride) {   // e0: the wavefront's first position (wave-uniform)
    const int64_t e = e0 + lane;
    int64_t k = -1, kp = -1;
    if (e < n) {
      k = static_cast<int64_t>(keys[e]);
      if (e > 0) kp = static_cast<int64_t>(keys[e - 1]);
      if (k > num_src) k = num_src;    // keys beyond the bound have no offset of their own
      if (kp > num_src) kp = num_src;
    }
    const int64_t gap = k - kp;        // entries (kp, k] hold e
    if (gap > 0 && gap <= kIndptrShortGap)
      for (int64_t t = kp + 1; t <= k; ++t) csr_indptr[t] = e;
    uint64_t wide = ballot(gap > kIndptrShortGap);
    while (wide != 0) {
      const int src = __ffsll(static_cast<long long>(wide)) - 1;
      wide &= wide - 1;
      const int64_t a = __shfl(kp, src, kWave) + 1, b = __shfl(k, src, kWave);
      for (int64_t t = a + lane; t <= b; t += kWave) csr_indptr[t] = e0 + src;
    }
  }
  for (int64_t t = last + 1 + tid; t <= num_src; t += stride) csr_indptr[t] = n;
}

// An empty block: offsets all zero.
__global__ __launch_bounds__(kFmtBlock) void fmt_zero_kernel(int64_t* a, int64_t na, int64_t* b, int64_t nb,
                                                             int64_t* c) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kFmtBlock + threadIdx.x; i < na || i < nb;
       i += static_cast<int64_t>(gridDim.x) * kFmtBlock) {
    if (a != nullptr && i < na) a[i] = 0;
    if (b != nullptr && i < nb) b[i] = 0;
  }
  if (c != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *c = 0;
}

int tuning_block_fused_scan();  // 0 = always take the separate scan launches

static size_t fmt_align(size_t x) { return (x + 255) / 256 * 256; }

struct FmtLayout {
  int64_t slots, ctiles, stiles, rtiles;
  size_t tile_cnt_off, sums_off, hist_off, bin_total_off, key_off[2], pay_off[2], total;
  int range_shift2, ranges;   // CSR by source ranges; ranges == 0: by radix passes
  size_t start_off, rec_off, part0_off, part_range_off, part_keys_off;
};

// Keys of the widest of so many ranges.
static int range_keys(int64_t ranges, int shift2) {
  return 1 << (ranges > kRangeCount0 + kRangeCount1 ? shift2 : ranges > kRangeCount0 ? kRangeShift1 : kRangeShift0);
}
// Long ranges have more than kRangeLong = 2 kRangePart records each: at most 3 parts to 2 kRangePart records.
static int64_t most_parts(int64_t slots) { return 3 * slots / (2 * kRangePart) + 1; }
static_assert(kRangeLong >= 2 * kRangePart && kRangePart % kRangeSortChunk == 0);

// The last piece's ranges are as narrow as their number allows.  num_src itself has a range: the last offset.
// A block of so few sources that every range is long is better off with the radix passes, of which it needs one or two:
// 1 M edges of 31 / 1000 / 2000 / 4000 sources, radix 42 / 70 / 69 / 69, ranges 40 / 95 / 106 / 61 us.  (The transpose has no
// radix passes.)
constexpr int64_t kRangeMostMean = 3000;
static void choose_ranges(int64_t num_dst, int64_t num_src, bool records_hold_dst, FmtLayout& L) {
  L.range_shift2 = kRangeShift2;
  while (L.range_shift2 < kRangeMaxShift && range_index(num_src, L.range_shift2) >= kRangeMaxCount) ++L.range_shift2;
  const int64_t ranges = range_index(num_src, L.range_shift2) + 1;
  const bool fits = ranges <= kRangeMaxCount && L.ctiles <= kRangeMaxTiles &&
                    (!records_hold_dst || (num_dst <= kRangeMaxDst &&
                                           (num_src >= kRangeFrom1 || L.slots <= kRangeMostMean * ranges))) &&
                    tuning_block_fused_scan();
  L.ranges = fits ? static_cast<int>(ranges) : 0;
}

static void lay_out_ranges(size_t off, int64_t tiles, int64_t ranges, int64_t slots, FmtLayout& L) {
  L.rtiles = tiles;
  L.tile_cnt_off = off;  off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(tiles));
  L.hist_off = off;      off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(tiles) * ranges);
  L.bin_total_off = off; off = fmt_align(off + sizeof(uint32_t) * ranges);
  L.start_off = off;     off = fmt_align(off + sizeof(uint32_t) * (ranges + 1));
  L.part0_off = off;     off = fmt_align(off + sizeof(uint32_t) * (ranges + 1));   // (and the number of parts)
  L.part_range_off = off; off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(most_parts(slots)));
  L.part_keys_off = off; off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(most_parts(slots)) * range_keys(ranges, L.range_shift2));
  L.rec_off = off;       L.total = fmt_align(off + sizeof(uint64_t) * static_cast<size_t>(slots));
}

static void lay_out_radix(size_t off, int64_t slots, FmtLayout& L) {
  L.hist_off = off;      off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(L.stiles) * kRadix);
  L.bin_total_off = off; off = fmt_align(off + sizeof(uint32_t) * kRadix);
  for (int k = 0; k < 2; ++k) {
    L.key_off[k] = off; off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(slots));
    L.pay_off[k] = off; off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(slots));
  }
  L.total = off;
}

static FmtLayout fmt_layout(int64_t num_dst, int fanout, int64_t num_src, bool csr, bool transpose = false) {
  FmtLayout L;
  L.ranges = 0;
  L.rtiles = 0;
  L.slots = num_dst * fanout;
  const int64_t slots = std::max<int64_t>(L.slots, 1);
  L.ctiles = ceil_div(slots, kCompactTile);
  L.stiles = ceil_div(slots, kSortTile);
  size_t off = 0;
  L.tile_cnt_off = off; off = fmt_align(off + sizeof(uint32_t) * static_cast<size_t>(L.ctiles));
  L.sums_off = off;     off = fmt_align(off + sizeof(uint32_t) * kScanChunk);
  L.total = L.hist_off = off;
  if (!csr) return L;
  choose_ranges(num_dst, num_src, !transpose, L);
  // ranges: by either tile, which one is the launch's choice
  if (L.ranges > 0)
    lay_out_ranges(off, slots <= kRangeSmallBound ? ceil_div(slots, kFmtBlock * kRangeSmallIters) : L.ctiles, L.ranges, slots, L);
  else
    lay_out_radix(off, slots, L);
  return L;
}

// What a block within these bounds takes at the most: a caller may size one workspace for its largest block.  A smaller
// block can have more ranges (narrower ones), more tiles (shorter ones) or other passes than the largest.
static size_t fmt_workspace(int64_t num_dst, int fanout, int64_t num_src, bool csr, bool transpose = false) {
  const FmtLayout L = fmt_layout(num_dst, fanout, num_src, csr, transpose);
  if (!csr) return L.total;
  const int64_t slots = std::max<int64_t>(L.slots, 1);
  FmtLayout most = L;
  const int64_t tiles = std::max(ceil_div(std::min(slots, kRangeSmallBound), kFmtBlock * kRangeSmallIters),
                                 std::min(L.ctiles, kRangeMaxTiles));
  const size_t head = fmt_align(sizeof(uint32_t) * static_cast<size_t>(L.ctiles)) + fmt_align(sizeof(uint32_t) * kScanChunk);
  lay_out_ranges(head, tiles, std::min<int64_t>(range_index(num_src, kRangeShift2) + 1, kRangeMaxCount),
                 std::min(slots, kRangeMaxTiles * kCompactTile), most);
  size_t total = std::max(L.total, most.total);
  if (!transpose) {
    lay_out_radix(head, slots, most);
    total = std::max(total, most.total);
  }
  return total;
}

static bool fmt_sizes_ok(int64_t num_dst, int fanout, int64_t num_src) {
  return num_dst >= 0 && fanout >= 0 && num_src >= 0 && num_src <= 0xffffffffLL &&
         (fanout == 0 || num_dst <= 0x7fffffffLL / fanout);
}

template <bool FORMATS>
static int launch_ranges(const CompactParams& c, RangeParams& r, const FmtLayout& L, char* ws, int64_t num_src,
                         hipStream_t st) {
  r.shift2 = L.range_shift2;
  r.ranges = L.ranges;
  r.hist = reinterpret_cast<uint32_t*>(ws + L.hist_off);
  r.total = reinterpret_cast<uint32_t*>(ws + L.bin_total_off);
  r.start = reinterpret_cast<uint32_t*>(ws + L.start_off);
  r.part0 = reinterpret_cast<uint32_t*>(ws + L.part0_off);
  r.parts = r.part0 + L.ranges;
  r.part_range = reinterpret_cast<uint32_t*>(ws + L.part_range_off);
  r.part_keys = reinterpret_cast<uint32_t*>(ws + L.part_keys_off);
  r.rec = reinterpret_cast<uint64_t*>(ws + L.rec_off);
  r.num_src = num_src;
  const int keys = r.row_words = range_keys(L.ranges, L.range_shift2);
  r.long_from = static_cast<uint32_t>(std::min<int64_t>(std::max<int64_t>(kRangeLong, 4 * L.slots / L.ranges), kRangeLongest));
  r.part_groups = L.slots > r.long_from ? static_cast<int>(std::min<int64_t>(ceil_div(L.slots, kRangePart), kRangePartGroups)) : 0;
  const bool small = L.slots <= (c.num_dst_dev != nullptr ? kRangeSmallBound : kRangeSmallSlots);
  r.tile = small ? kFmtBlock * kRangeSmallIters : kCompactTile;
  const dim3 tiles(static_cast<unsigned>(ceil_div(std::max<int64_t>(L.slots, 1), r.tile)));
  const size_t count_lds = sizeof(uint32_t) * L.ranges;
  if (small)
    hipLaunchKernelGGL((range_count_kernel<FORMATS, kRangeSmallIters>), tiles, dim3(kFmtBlock), count_lds, st, c, r);
  else
    hipLaunchKernelGGL((range_count_kernel<FORMATS, kCompactIters>), tiles, dim3(kFmtBlock), count_lds, st, c, r);
  APT_LAUNCH_CHECK("range_count_kernel");
  hipLaunchKernelGGL(range_scan_kernel, dim3(static_cast<unsigned>(ceil_div(L.ranges, kWave))),
                     dim3(kWave * kRangeScanGroups), 0, st, c, r);
  APT_LAUNCH_CHECK("range_scan_kernel");
  const size_t place_lds = sizeof(uint32_t) * (L.ranges + kFmtWaves * ((L.ranges + 1) / 2));
  if (small)
    hipLaunchKernelGGL((range_place_kernel<FORMATS, kRangeSmallIters>), tiles, dim3(kFmtBlock), place_lds, st, c, r);
  else
    hipLaunchKernelGGL((range_place_kernel<FORMATS, kCompactIters>), tiles, dim3(kFmtBlock), place_lds, st, c, r);
  APT_LAUNCH_CHECK("range_place_kernel");
  hipLaunchKernelGGL(range_sort_kernel<FORMATS>, dim3(static_cast<unsigned>(r.part_groups + L.ranges)), dim3(kRangeSortBlock),
                     sizeof(uint32_t) * (keys + kRangeSortWaves * (keys / 2)), st, r);
  APT_LAUNCH_CHECK("range_sort_kernel");
  return APT_OK;
}

}  // namespace apt

extern "C" size_t apt_block_transpose_workspace_bytes(int64_t num_dst, int fanout, int64_t num_src) {
  using namespace apt;
  if (!fmt_sizes_ok(num_dst, fanout, num_src)) return 0;
  return fmt_layout(num_dst, fanout, num_src, true, true).ranges > 0 ? fmt_workspace(num_dst, fanout, num_src, true, true) : 0;
}

extern "C" int apt_block_transpose(const int64_t* relabeled, int64_t num_dst, int fanout, int64_t num_src,
                                   uint32_t* indptr, uint32_t* slots, void* long_table, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(fmt_sizes_ok(num_dst, fanout, num_src), APT_ELIMIT,
              "apt_block_transpose: sizes out of range (num_dst %lld, fanout %d, num_src %lld)",
              static_cast<long long>(num_dst), fanout, static_cast<long long>(num_src));
  const FmtLayout L = fmt_layout(num_dst, fanout, num_src, true, true);
  APT_REQUIRE(L.ranges > 0, APT_ELIMIT, "apt_block_transpose: block too large (see apt_block_transpose_workspace_bytes)");
  APT_REQUIRE(indptr != nullptr && (L.slots == 0 || (relabeled != nullptr && slots != nullptr)), APT_EINVAL,
              "apt_block_transpose: an argument is NULL");
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= L.total, APT_EWORKSPACE,
              "apt_block_transpose: workspace of %zu bytes, %zu needed", workspace_bytes, L.total);
  CompactParams c{};
  c.relabeled = relabeled;
  c.num_dst = num_dst;
  c.num_dst_dev = nullptr;
  c.fanout = fanout;
  c.tiles = L.ctiles;
  RangeParams r{};
  r.t_indptr = indptr;
  r.t_slots = slots;
  r.lng = long_rows(long_table, L.slots, nullptr);
  return launch_ranges<false>(c, r, L, static_cast<char*>(workspace), num_src, static_cast<hipStream_t>(stream));
}

extern "C" size_t apt_block_workspace_bytes(int64_t num_dst, int fanout, int64_t num_src, int want_csr) {
  using namespace apt;
  if (!fmt_sizes_ok(num_dst, fanout, num_src)) return 0;
  return fmt_workspace(num_dst, fanout, num_src, want_csr != 0);
}

extern "C" int apt_block_formats(const int64_t* relabeled, int64_t num_dst, const int64_t* num_dst_dev,
                                 int fanout, int64_t num_src, int64_t* coo_row, int64_t* coo_col,
                                 int64_t* csc_indptr, int64_t* num_edges_dev, int64_t* csr_indptr,
                                 int64_t* csr_indices, int64_t* csr_eids, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(fmt_sizes_ok(num_dst, fanout, num_src), APT_ELIMIT,
              "apt_block_formats: sizes out of range (num_dst %lld, fanout %d, num_src %lld)",
              static_cast<long long>(num_dst), fanout, static_cast<long long>(num_src));
  APT_REQUIRE(csc_indptr != nullptr && num_edges_dev != nullptr, APT_EINVAL,
              "apt_block_formats: csc_indptr / num_edges_dev is NULL");
  const bool csr = csr_indptr != nullptr;
  APT_REQUIRE(!csr || (csr_indices != nullptr && csr_eids != nullptr), APT_EINVAL,
              "apt_block_formats: csr_indices / csr_eids is NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const FmtLayout L = fmt_layout(num_dst, fanout, num_src, csr);
  if (L.slots == 0) {
    const int64_t longest = std::max<int64_t>(num_dst + 1, csr ? num_src + 1 : 0);
    hipLaunchKernelGGL(fmt_zero_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(longest, kFmtBlock), 4096))),
                       dim3(kFmtBlock), 0, st, csc_indptr, num_dst + 1, csr_indptr, csr ? num_src + 1 : 0,
                       num_edges_dev);
    APT_LAUNCH_CHECK("fmt_zero_kernel");
    return APT_OK;
  }
  APT_REQUIRE(relabeled != nullptr && coo_row != nullptr && coo_col != nullptr, APT_EINVAL,
              "apt_block_formats: relabeled / coo_row / coo_col is NULL");
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= L.total, APT_EWORKSPACE,
              "apt_block_formats: workspace of %zu bytes, %zu needed", workspace_bytes, L.total);
  char* ws = static_cast<char*>(workspace);
  uint32_t* sums = reinterpret_cast<uint32_t*>(ws + L.sums_off);

  CompactParams c;
  c.relabeled = relabeled;
  c.num_dst = num_dst;
  c.num_dst_dev = num_dst_dev;
  c.fanout = fanout;
  c.tile_cnt = reinterpret_cast<uint32_t*>(ws + L.tile_cnt_off);
  c.coo_row = coo_row;
  c.coo_col = coo_col;
  c.csc_indptr = csc_indptr;
  c.tiles = L.ctiles;
  c.scanned = L.ctiles > kFusedCompactTiles || !tuning_block_fused_scan();
  c.num_edges_dev = num_edges_dev;
  const dim3 cgrid(static_cast<unsigned>(L.ctiles));
  if (L.ranges > 0) {
    RangeParams r{};
    r.csr_indptr = csr_indptr;
    r.csr_indices = csr_indices;
    r.csr_eids = csr_eids;
    return launch_ranges<true>(c, r, L, ws, num_src, st);
  }
  hipLaunchKernelGGL(fmt_count_kernel, cgrid, dim3(kFmtBlock), 0, st, c);
  APT_LAUNCH_CHECK("fmt_count_kernel");
  // the edge total is also the last CSC offset
  if (c.scanned)
    if (int rc = exclusive_scan(c.tile_cnt, L.ctiles, sums, num_edges_dev, csc_indptr + num_dst, st)) return rc;
  hipLaunchKernelGGL(fmt_place_kernel, cgrid, dim3(kFmtBlock), 0, st, c);
  APT_LAUNCH_CHECK("fmt_place_kernel");
  if (!csr) return APT_OK;

  int bits = 1;
  while (bits < 32 && (1LL << bits) < num_src) ++bits;
  const int passes = (bits + kRadixBits - 1) / kRadixBits;
  SortParams s;
  s.coo_row = coo_row;
  s.coo_col = coo_col;
  s.num_edges_dev = num_edges_dev;
  s.max_edges = L.slots;
  s.tile_hist = reinterpret_cast<uint32_t*>(ws + L.hist_off);
  s.bin_total = reinterpret_cast<uint32_t*>(ws + L.bin_total_off);
  s.tiles = L.stiles;
  s.fused = L.stiles <= kFusedSortTiles && tuning_block_fused_scan();
  s.csr_indices = csr_indices;
  s.csr_eids = csr_eids;
  const dim3 sgrid(static_cast<unsigned>(L.stiles));
  for (int pass = 0; pass < passes; ++pass) {
    const bool first = pass == 0, last = pass == passes - 1;
    s.shift = pass * kRadixBits;
    s.key_in = first ? nullptr : reinterpret_cast<uint32_t*>(ws + L.key_off[(pass - 1) & 1]);
    s.pay_in = first ? nullptr : reinterpret_cast<uint32_t*>(ws + L.pay_off[(pass - 1) & 1]);
    s.key_out = reinterpret_cast<uint32_t*>(ws + L.key_off[pass & 1]);
    s.pay_out = reinterpret_cast<uint32_t*>(ws + L.pay_off[pass & 1]);
    if (first) hipLaunchKernelGGL(radix_hist_kernel<true>, sgrid, dim3(kSortBlock), 0, st, s);
    else hipLaunchKernelGGL(radix_hist_kernel<false>, sgrid, dim3(kSortBlock), 0, st, s);
    APT_LAUNCH_CHECK("radix_hist_kernel");
    if (!s.fused) {
      hipLaunchKernelGGL(radix_binscan_kernel, dim3(kRadix), dim3(kSortBlock), 0, st, s);
      APT_LAUNCH_CHECK("radix_binscan_kernel");
    }
    if (first && last) hipLaunchKernelGGL((radix_scatter_kernel<true, true>), sgrid, dim3(kSortBlock), 0, st, s);
    else if (first) hipLaunchKernelGGL((radix_scatter_kernel<true, false>), sgrid, dim3(kSortBlock), 0, st, s);
    else if (last) hipLaunchKernelGGL((radix_scatter_kernel<false, true>), sgrid, dim3(kSortBlock), 0, st, s);
    else hipLaunchKernelGGL((radix_scatter_kernel<false, false>), sgrid, dim3(kSortBlock), 0, st, s);
    APT_LAUNCH_CHECK("radix_scatter_kernel");
  }
  const uint32_t* sorted = reinterpret_cast<uint32_t*>(ws + L.key_off[(passes - 1) & 1]);
  const unsigned iblocks =
      static_cast<unsigned>(std::min<int64_t>(ceil_div(std::max<int64_t>(num_src + 1, L.slots), kFmtBlock), 4096));
  hipLaunchKernelGGL(csr_indptr_kernel, dim3(iblocks), dim3(kFmtBlock), 0, st, sorted, num_edges_dev, L.slots,
                     num_src, csr_indptr);
  APT_LAUNCH_CHECK("csr_indptr_kernel");
  return APT_OK;
}

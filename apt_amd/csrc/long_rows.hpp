// Rows of a sum over grouped edges that are far longer than the others: a readout's few rows, a hub among the sources.
// One workgroup would add them up long after the others are done (1 M edges of 64 fp32 features into one row: 11.6 ms),
// so their edges are cut into chunks for many workgroups.  A chunk's sum goes to a buffer; the workgroup that finishes a
// row's last chunk adds them up in their order, so nobody waits and the result does not depend on who was last.  1 M edges
// of 64 fp32 (one workgroup a row / edge by edge with atomics / chunks, host reads included): into 1 row 11 680 / 1550 /
// 127 us, 8 rows 11 700 / 429 / 124, 64 rows 5940 / 148 / 136; half of them into one of 100 k rows 5700 / 829 / 111.
//
// A row is long if it has more than a 512th of all edges (a workgroup's share of a full launch is a 2048th), and more than
// kLongLeast.  The long rows of a launch are found before it: row r stands in slot offset(r) / `longer` of a table.  Two long
// rows never share one, since a row that begins after a long one begins more than `longer` edges later.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace apt {

constexpr int64_t kLongLeast = 512;
constexpr int64_t kLongShare = 512;
constexpr int64_t kLongChunk = 256;          // edges of a chunk: this many, half of `longer`, or a 1024th of the row
constexpr int64_t kLongMostChunks = 1024;

struct LongRows {
  uint32_t* row;        // [slots]: row + 1, 0 = none
  uint32_t* arrived;    // [slots]: finished chunks, 0 between launches
  float* part;          // [chunks][width]
  int slots;            // 0: no row is long
  uint32_t longer;      // a row of more edges is long
  uint32_t chunk;       // edges of a chunk at least
};

inline int64_t long_from(int64_t num_edges) { return std::max(kLongLeast, ceil_div(num_edges, kLongShare)); }
inline int64_t long_slots(int64_t num_edges) { return num_edges > kLongLeast ? num_edges / long_from(num_edges) + 1 : 0; }
inline int64_t long_chunk(int64_t num_edges) { return std::max(kLongChunk, long_from(num_edges) / 2); }
// A long row of n edges has at most n / long_chunk + 1 <= 3 n / long_from chunks (long_from + 1 >= 2 long_chunk).
inline int64_t long_chunks(int64_t num_edges) { return num_edges > kLongLeast ? 3 * num_edges / long_from(num_edges) + 1 : 0; }

inline LongRows long_rows(void* table, int64_t num_edges, float* part) {
  LongRows l{};
  if (table == nullptr || long_slots(num_edges) == 0) return l;
  l.slots = static_cast<int>(long_slots(num_edges));
  l.row = static_cast<uint32_t*>(table);
  l.arrived = l.row + l.slots;
  l.part = part;
  l.longer = static_cast<uint32_t>(long_from(num_edges));
  l.chunk = static_cast<uint32_t>(long_chunk(num_edges));
  return l;
}

// The chunks as one workgroup sees them.  They are numbered by thread: thread t speaks for every BLOCK-th slot.
template <int BLOCK, typename I>
struct LongChunks {
  const LongRows& l;
  const I* indptr;
  uint32_t from = 0, to = 0;   // the thread's
  uint32_t all = 0;
  __device__ __forceinline__ LongChunks(const LongRows& rows, const I* offsets) : l(rows), indptr(offsets) {}
  __device__ __forceinline__ uint32_t length(uint32_t n) const {
    return max(l.chunk, static_cast<uint32_t>((n + kLongMostChunks - 1) / kLongMostChunks));
  }
  __device__ __forceinline__ uint32_t chunks_of(int slot) const {
    const uint32_t row = l.row[slot];
    if (row == 0) return 0;
    const uint32_t n = static_cast<uint32_t>(indptr[row] - indptr[row - 1]);
    return (n + length(n) - 1) / length(n);
  }
  // For the whole workgroup; s_wave: [BLOCK / kWave]
  __device__ __forceinline__ void number(uint32_t* s_wave) {
    uint32_t mine = 0;
    for (int s = threadIdx.x; s < l.slots; s += BLOCK) mine += chunks_of(s);
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    uint32_t incl = mine;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    all = 0;
    for (int w = 0; w < BLOCK / kWave; ++w) {
      if (w < wave) before += s_wave[w];
      all += s_wave[w];
    }
    to = before + incl;
    from = to - mine;
  }
  struct Chunk {
    int slot;
    int64_t row, from, to;    // edges
    uint32_t index, count;    // its number in the row, and the row's chunks
  };
  // Chunk p, for the whole workgroup; s_where: [2]
  __device__ __forceinline__ Chunk find(uint32_t p, uint32_t* s_where) const {
    __syncthreads();   // (the last chunk's place has been read)
    if (p >= from && p < to) {
      uint32_t run = from;
      for (int s = threadIdx.x; s < l.slots; s += BLOCK) {
        const uint32_t has = chunks_of(s);
        if (p - run < has) {
          s_where[0] = static_cast<uint32_t>(s);
          s_where[1] = p - run;
          break;
        }
        run += has;
      }
    }
    __syncthreads();
    Chunk c;
    c.slot = static_cast<int>(s_where[0]);
    c.index = s_where[1];
    c.row = static_cast<int64_t>(l.row[c.slot]) - 1;
    const int64_t lo = static_cast<int64_t>(indptr[c.row]), hi = static_cast<int64_t>(indptr[c.row + 1]);
    const uint32_t len = length(static_cast<uint32_t>(hi - lo));
    c.count = (static_cast<uint32_t>(hi - lo) + len - 1) / len;
    c.from = lo + static_cast<int64_t>(c.index) * len;
    c.to = min(c.from + len, hi);
    return c;
  }
  // The workgroup has stored the chunk's sum: whether it was the last of its row.  If so, all of the row's sums can be read.
  __device__ __forceinline__ bool last_of_row(const Chunk& c, uint32_t* s_last) const {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // (vmcnt(0): every wavefront's stores are in the L2 before thread 0 writes it back)
    __syncthreads();
    if (threadIdx.x == 0) {
      __threadfence();   // the workgroup's stores before the count, the other workgroups' behind it
      const uint32_t n = atomicAdd(&l.arrived[c.slot], 1u) + 1;
      if (n == c.count) l.arrived[c.slot] = 0;   // (for the next launch on this table)
      *s_last = n == c.count;
      __threadfence();
    }
    __syncthreads();
    return *s_last != 0;
  }
};

}  // namespace apt

// Gradients of dense layers' weights and biases over the rows of a block:
//   dw[n, k] = sum_m dy[m, n] * x[m, k],   db[n] = sum_m dy[m, n]
// for one or two such products in one launch (a GraphSAGE layer has two, a GCN layer one and the column sums of
// another matrix); dy may still need the mask of the ReLU that it passed.
//
// A block has 10^4..10^6 rows and a layer a few hundred columns, so a product reduces over the one long dimension
// and its output is a few tiles.  The rows are split over the chip, a workgroup accumulates one output tile of its
// rows in MFMA accumulators and leaves it in a partial buffer, and a second launch adds the partials in a fixed
// order (reproducible, no atomics).
//
// fp32 operands are multiplied as bf16 parts (split_bf16.hpp): the fp32 matrix instruction would bound the product.
// Splitting costs as many cycles of the vector units as its six products cost the matrix units, so a step's rows
// are split once, into LDS, and read from there by all wavefronts that need them.  Both operands have the reduced
// dimension as their row index, which is what an MFMA operand wants *inside* a lane (8 consecutive rows of one
// column): a thread loads 8 rows of a few columns and regroups them by column on the way into LDS.
#include <algorithm>

#include "common.hpp"
#include "feature_rows.hpp"
#include "split_bf16.hpp"

namespace apt {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// Buffer loads: a range-checked base in scalar registers plus a 32-bit lane offset; what lies past the range reads
// as zero, so neither the last rows of a split nor the columns past the edge of a tile need a branch.
typedef uint32_t u32x2_v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_v __attribute__((ext_vector_type(4)));
using buffer_t = __amdgpu_buffer_rsrc_t;

// It begins at a multiple of four bytes (`skip`: how far behind that the base is) and ends at one.
__device__ __forceinline__ buffer_t make_buffer(const void* base, int64_t bytes, uint32_t& skip) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(base);
  skip = static_cast<uint32_t>(at & 3);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at - skip), 0,
                                           bytes > 0 ? static_cast<uint32_t>(bytes + skip + 3) & ~3u : 0u, 0x00020000);
}

constexpr int kWgradWaves = 4;      // that multiply, two by two; as many more prepare their operands
constexpr int kWgradHalf = kWgradWaves * kWave;
constexpr int kWgradBlock = 2 * kWgradHalf;
constexpr int kWgradGroups = 256;   // workgroups aimed at: one per CU ...
constexpr int kWgradSmallGroups = 512;   // ... or, of smaller tiles, two while each has kWgradSmallSteps of its loop
constexpr int kWgradSmallSteps = 16;
constexpr int64_t kWgradLongRows = 1 << 19;   // times tiles: from here on oblong ones (see wgrad_shape)
constexpr int kWgradJobs = 2;
constexpr int64_t kWgradPartBytes = int64_t{16} << 20;

struct WgradJob {
  const void* dy;      // [m, n]
  const void* out;     // [m, n] or NULL: dy counts where out > 0
  const void* x;       // [m, k]; k == 0: the column sums alone
  int64_t m, n, k;
  float* part;         // [splits][stride]: dw, then db
  int64_t stride;
  int tiles_k, tiles;  // output tiles: tiles_n * tiles_k
  int splits;
  void *dw, *db;
};

struct WgradParams {
  WgradJob job[kWgradJobs];
  int jobs, tiles;          // of all jobs
  int common, longer;       // splits that all jobs have; the job that has more
  int groups;               // workgroups
  int64_t rows_per_split;
};

// Rows of a step and how a thread reads them: a unit is 8 rows (one lane's share of an MFMA operand) of kCols columns.
// WgradOdd: bf16 rows of an odd length or address; a dword more is read, and the elements are taken out of the three.
// WgradRelu: products may have a mask.
struct WgradOdd {};
template <typename T> struct WgradRelu {};
template <typename T> struct WgradType;
template <> struct WgradType<float> {
  using Elem = float;
  static constexpr int kRows = 32, kCols = 2, kWords = 2, kParts = 3;
  static constexpr bool kMask = false;
};
template <> struct WgradType<uint16_t> {
  using Elem = uint16_t;
  static constexpr int kRows = 64, kCols = 4, kWords = 2, kParts = 1;
  static constexpr bool kMask = false;
};
template <> struct WgradType<WgradOdd> : WgradType<uint16_t> {
  static constexpr int kWords = 3;
};
template <typename T> struct WgradType<WgradRelu<T>> : WgradType<T> {
  static constexpr bool kMask = true;
};
constexpr int kUnitRows = 8;
constexpr int kWgradAhead = 2;   // steps whose rows are on their way
// Where column c of a fragment stands in LDS, and the reverse: a thread's columns are apart from each other, those of its
// neighbours together, so that a store of a wavefront meets every bank alike.  The lanes of an operand have the columns in
// this order.
template <typename T> __host__ __device__ constexpr int wgrad_place(int c) {
  return c % WgradType<T>::kCols * (16 / WgradType<T>::kCols) + c / WgradType<T>::kCols;
}
template <typename T> __host__ __device__ constexpr int wgrad_col(int place) {
  return place % (16 / WgradType<T>::kCols) * WgradType<T>::kCols + place / (16 / WgradType<T>::kCols);
}
// A workgroup's output tile, 2 FN x 2 FK fragments, and its LDS: a step's operands twice, and the column sums.
template <typename T, int FN, int FK> struct WgradTile {
  static constexpr int kTileN = 2 * FN * 16, kTileK = 2 * FK * 16;
  static constexpr int kGroups = WgradType<T>::kRows / kUnitRows;
  static constexpr int kBuffer = WgradType<T>::kParts * WgradType<T>::kRows * (kTileN + kTileK) * 2;
  static constexpr int kLds = 2 * kBuffer + kGroups * kTileN * 4;
};

template <typename T> struct WgradUnit {
  using Type = WgradType<T>;
  uint32_t v[kUnitRows][Type::kWords];
  // (no choice between kinds of loads here: registers that two branches load are moved, and waited for, behind them.
  // Every dword of a load has a range check of its own.)
  __device__ __forceinline__ void load(buffer_t buf, uint32_t at, uint32_t row_bytes) {
#pragma unroll
    for (int r = 0; r < kUnitRows; ++r, at += row_bytes) {
      const uint32_t from = Type::kWords == 3 ? at & ~3u : at;
      const u32x2_v w = __builtin_amdgcn_raw_buffer_load_b64(buf, from, 0, 0);
      v[r][0] = w[0];
      v[r][1] = w[1];
      if constexpr (Type::kWords == 3) v[r][2] = __builtin_amdgcn_raw_buffer_load_b32(buf, from + 8, 0, 0);
    }
  }
  // Elements where the even ones of the other kind are.  odd_at: the first row begins in the middle of a dword; odd_row: so does
  // every other row.
  __device__ __forceinline__ void align(uint32_t odd_at, uint32_t odd_row) {
    if constexpr (Type::kWords == 3) {
#pragma unroll
      for (int r = 0; r < kUnitRows; ++r) {
        const uint32_t shift = 16 * ((odd_at ^ (r & odd_row)) & 1);
        v[r][0] = __builtin_amdgcn_alignbit(v[r][1], v[r][0], shift);
        v[r][1] = __builtin_amdgcn_alignbit(v[r][2], v[r][1], shift);
      }
    }
  }
  // The first element of a row is none: what shares a dword with the last of the range.
  __device__ __forceinline__ void drop_first(int row) {
#pragma unroll
    for (int r = 0; r < kUnitRows; ++r) v[r][0] &= r == row ? 0xffff0000u : 0xffffffffu;
  }
  // Zero where the ReLU's result is (as torch has it: a NaN passes).
  __device__ __forceinline__ void mask(const WgradUnit& out) {
#pragma unroll
    for (int r = 0; r < kUnitRows; ++r)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if constexpr (Type::kParts == 3) {
          v[r][w] = __uint_as_float(out.v[r][w]) <= 0.f ? 0u : v[r][w];
        } else {
          const uint32_t lo = __uint_as_float(out.v[r][w] << 16) <= 0.f ? 0u : 0xffffu;
          const uint32_t hi = __uint_as_float(out.v[r][w] & 0xffff0000u) <= 0.f ? 0u : 0xffff0000u;
          v[r][w] &= lo | hi;
        }
      }
  }
  __device__ __forceinline__ void add_to(float (&sum)[Type::kCols]) const {
#pragma unroll
    for (int c = 0; c < Type::kCols; ++c) {
      float even = 0.f, odd = 0.f;
#pragma unroll
      for (int r = 0; r < kUnitRows; r += 2) {
        if constexpr (Type::kParts == 3) {
          even += __uint_as_float(v[r][c]);
          odd += __uint_as_float(v[r + 1][c]);
        } else {
          even += __uint_as_float((c & 1) != 0 ? v[r][c / 2] & 0xffff0000u : v[r][c / 2] << 16);
          odd += __uint_as_float((c & 1) != 0 ? v[r + 1][c / 2] & 0xffff0000u : v[r + 1][c / 2] << 16);
        }
      }
      sum[c] += even + odd;
    }
  }
  // Column c of the unit as MFMA operand: eight bf16 (per part), two rows to a register.
  __device__ __forceinline__ void column(int c, u32x4_v (&o)[Type::kParts]) const {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if constexpr (Type::kParts == 3) {
        const SplitPair s = split_pair(__uint_as_float(v[2 * d][c]), __uint_as_float(v[2 * d + 1][c]));
        o[0][d] = s.hi;
        o[1][d] = s.mid;
        o[2][d] = s.lo;
      } else {
        o[0][d] = __builtin_amdgcn_perm(v[2 * d + 1][c / 2], v[2 * d][c / 2], (c & 1) != 0 ? 0x07060302u : 0x05040100u);
      }
    }
  }
};

__device__ __forceinline__ f32x4_t wgrad_mfma(u32x4_v a, u32x4_v b, f32x4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}

// FN x FK fragments (of 16 x 16 outputs) per wavefront.  Four wavefronts read the rows, split them and leave them in LDS
// (producers), the other four multiply what the step before left there (consumers): with one of either on a SIMD the
// vector units and the matrix units work at the same time.
template <typename T, int FN, int FK>
__global__ __launch_bounds__(kWgradBlock) void wgrad_kernel(WgradParams p) {
  using Type = WgradType<T>;
  using Elem = typename Type::Elem;
  using Tile = WgradTile<T, FN, FK>;
  constexpr int kRows = Type::kRows, kCols = Type::kCols, kParts = Type::kParts;
  constexpr int kGroups = Tile::kGroups, kSubs = kRows / 32;
  constexpr int kTileN = Tile::kTileN, kTileK = Tile::kTileK;
  constexpr int kUnitsN = kTileN / kCols * kGroups, kUnitsK = kTileK / kCols * kGroups;   // of dy and of x
  constexpr int kUnits = FN + FK > 4 ? 2 : 1;                     // of a producer: 2 = one of either, 1 = of dy or of x
  static_assert(std::max(kUnitsN, kUnitsK) * 2 == kUnits * kWgradHalf && std::min(kUnitsN, kUnitsK) % kWave == 0);
  constexpr int kFrags = 2 * FN + 2 * FK;                         // of the tile's operands: dy's, then x's
  constexpr int kFlip = kCols == 4 ? 4 : 0;                       // four lanes to a fragment: its neighbour the other way round
  static_assert(kWgradAhead % 2 == 0 && FN % 2 == 0);
  extern __shared__ __align__(16) char s_wgrad[];
  u32x4_v* s_part = reinterpret_cast<u32x4_v*>(s_wgrad);          // [buffer][part][sub][fragment][lane]
  float(*s_sum)[kTileN] = reinterpret_cast<float(*)[kTileN]>(s_wgrad + 2 * Tile::kBuffer);
  constexpr int kBufferVecs = Tile::kBuffer / 16, kPartVecs = kBufferVecs / kParts;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = lane / 16, col16 = wgrad_col<T>(lane % 16);
  // The workgroups of a split read the same rows: they follow each other on one XCD, whose L2 then serves the others.  First
  // the splits that all products have, then the others of the longer one.
  const int w = static_cast<int>(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8);
  if (w >= p.groups) return;   // block-uniform
  const bool common = w < p.common * p.tiles;
  const int in = common ? w : w - p.common * p.tiles, tiles = common ? p.tiles : p.job[p.longer].tiles;
  const int split = __builtin_amdgcn_readfirstlane(in / tiles + (common ? 0 : p.common));   // (a division leaves them in
  int tile = __builtin_amdgcn_readfirstlane(in % tiles);                                    // vector registers)
  const int which = common ? (p.jobs > 1 && tile >= p.job[0].tiles ? 1 : 0) : p.longer;
  const WgradJob& job = p.job[which];
  if (common && which == 1) tile -= p.job[0].tiles;
  const int tile_n = __builtin_amdgcn_readfirstlane(tile / job.tiles_k), tile_k = tile - tile_n * job.tiles_k;
  const int64_t n0 = static_cast<int64_t>(tile_n) * kTileN, k0 = static_cast<int64_t>(tile_k) * kTileK;
  const int64_t m0 = static_cast<int64_t>(split) * p.rows_per_split;
  const int64_t m1 = min(m0 + p.rows_per_split, job.m);
  const bool bias = job.db != nullptr && tile_k == 0;
  const bool masked = job.out != nullptr;
  uint32_t skip_a, skip_out, skip_b;
  const buffer_t dy = make_buffer(static_cast<const Elem*>(job.dy) + m0 * job.n, (m1 - m0) * job.n * sizeof(Elem), skip_a);
  const buffer_t out = make_buffer(static_cast<const Elem*>(masked ? job.out : job.dy) + m0 * job.n,
                                   (m1 - m0) * job.n * sizeof(Elem), skip_out);
  const buffer_t x = make_buffer(static_cast<const Elem*>(job.x) + m0 * job.k, (m1 - m0) * job.k * sizeof(Elem), skip_b);
  // (whole turns of the producers' loop; a step past the end reads zeros)
  const int steps = static_cast<int>((m1 - m0 + kWgradAhead * kRows - 1) / (kWgradAhead * kRows)) * kWgradAhead;

  const int wn = (wave & 3) / 2, wk = wave % 2;
  const int64_t wave_n = n0 + wn * FN * 16, wave_k = k0 + wk * FK * 16;
  const bool active = wave < kWgradWaves && wave_n < job.n && wave_k < job.k;   // wave-uniform
  f32x4_t acc[FN][FK] = {};
  if (wave >= kWgradWaves) {
    // A thread's units: columns kCols * (u % units per row), rows 8 * (u / units per row) of a step.  Columns past the
    // edge read the row after (or zero): they only reach outputs past the edge, which are not stored.
    // The narrow side of a tile that is not square has units for two of the wavefronts: of either pair in turn, since the
    // workgroups of a CU come 256 apart and each has a wavefront on every SIMD.
    const int pair = FN != FK && (wave / 2 & 1) != (blockIdx.x / kWgradGroups & 1) ? 1 : 0;      // wave-uniform; 1: none
    const int thread = threadIdx.x - kWgradHalf, in_pair = threadIdx.x % (2 * kWave);
    const bool has_dy = kUnits == 2 ? FN >= FK || pair == 0 : wave - kWgradWaves < kUnitsN / kWave;   // wave-uniform
    const bool has_x = kUnits == 2 ? FN <= FK || pair == 0 : !has_dy;
    // A range that ends in the middle of a dword holds an element too many, the first of the row behind it: in step `end`, if
    // that is read at all.  (Its row and step in the range are the same for both operands.)
    const int rows = static_cast<int>(m1 - m0), end = rows / kRows;
    struct Source {
      buffer_t buffer;
      uint32_t row, at;
      int col, rg, frag0;
      uint32_t odd_at, odd_row;
      bool cut;      // of this thread's unit
    } source[kUnits];
    const auto operand = [&](buffer_t buffer, int64_t cols, int64_t col0, int u, int tile_cols, int frag0, uint32_t skip, bool here) {
      const int col = u % (tile_cols / kCols) * kCols, rg = u / (tile_cols / kCols);
      const uint32_t row = static_cast<uint32_t>(cols * sizeof(Elem));
      // (a unit of another wavefront's is read past the range)
      const uint32_t at = here ? static_cast<uint32_t>((rg * kUnitRows * cols + col0 + col) * sizeof(Elem)) + skip : 0x80000000u;
      return Source{buffer, here ? row : 0u, at, col, rg, frag0, skip >> 1, row >> 1 & 1,
                    col0 + col == 0 && rows % kRows / kUnitRows == rg && ((rows * cols * 2 + skip) & 2) != 0};
    };
    const Source a = operand(dy, job.n, n0, kUnits == 1 ? thread % kUnitsN : FN >= FK ? thread : in_pair, kTileN, 0, skip_a, has_dy);
    const Source b = operand(x, job.k, k0, kUnits == 1 ? thread % kUnitsK : FN <= FK ? thread : in_pair, kTileK, 2 * FN, skip_b, has_x);
    source[0] = kUnits == 2 || has_dy ? a : b;
    if constexpr (kUnits == 2) source[1] = b;
    const bool sum_here = bias && has_dy;
    WgradUnit<T> unit[kWgradAhead][kUnits], relu[kWgradAhead];
    auto load = [&](int q) {
      if constexpr (Type::kMask) relu[q].load(has_dy ? out : x, source[0].at + (has_dy ? skip_out - skip_a : 0u), source[0].row);
#pragma unroll
      for (int i = 0; i < kUnits; ++i) {
        unit[q][i].load(source[i].buffer, source[i].at, source[i].row);
        source[i].at += kRows * source[i].row;
      }
      __builtin_amdgcn_sched_barrier(0);   // (in this order: the first step's are waited for alone)
    };
    float sum[kCols] = {};
#pragma unroll
    for (int q = 0; q < kWgradAhead; ++q) load(q);
    for (int s = 0; s < steps; s += kWgradAhead) {
#pragma unroll
      for (int q = 0; q < kWgradAhead; ++q) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
          if (FN < FK && i == 0 && !has_dy) continue;   // (wave-uniform)
          if (FN > FK && i == 1 && !has_x) continue;
          WgradUnit<T> now = unit[q][i];
          now.align(source[i].odd_at, source[i].odd_row);
          if constexpr (Type::kMask) {
            if (i == 0 && masked && has_dy) {
              WgradUnit<T> result = relu[q];
              result.align(skip_out >> 1, source[0].odd_row);
              now.mask(result);
            }
          }
          if (Type::kWords == 3 && s + q == end && source[i].cut) now.drop_first(rows % kUnitRows);
          if (i == 0 && sum_here) now.add_to(sum);
#pragma unroll
          for (int c = 0; c < kCols; ++c) {
            u32x4_v o[kParts];
            now.column(c, o);
            const int col = source[i].col, rg = source[i].rg, frag = source[i].frag0 + col / 16;
            const int at = (q & 1) * kBufferVecs + ((rg / 4 * kFrags + frag) * 4 + rg % 4) * 16 + (wgrad_place<T>(col % 16 + c) ^ (frag & 1) * kFlip);
#pragma unroll
            for (int d = 0; d < kParts; ++d) s_part[d * kPartVecs + at] = o[d];
          }
        }
        load(q);
        __syncthreads();   // (one per step, of the producers and of the consumers)
      }
    }
    if (sum_here)
#pragma unroll
      for (int q = 0; q < kCols; ++q) s_sum[source[0].rg][source[0].col + q] = sum[q];
  } else {
    for (int s = 0; s < steps; ++s) {
      __syncthreads();
      if (!active) continue;
      const u32x4_v* from[2] = {s_part + (s & 1) * kBufferVecs + lane, s_part + (s & 1) * kBufferVecs + (lane ^ kFlip)};
#pragma unroll
      for (int h = 0; h < kSubs; ++h) {
        u32x4_v fa[FN][kParts];
#pragma unroll
        for (int f = 0; f < FN; ++f)
#pragma unroll
          for (int t = 0; t < kParts; ++t) fa[f][t] = from[f & 1][t * kPartVecs + (h * kFrags + wn * FN + f) * kWave];
#pragma unroll
        for (int g = 0; g < FK; ++g) {
          u32x4_v fb[kParts];
#pragma unroll
          for (int t = 0; t < kParts; ++t) fb[t] = from[g & 1][t * kPartVecs + (h * kFrags + 2 * FN + wk * FK + g) * kWave];
          // products of one accumulator are kept apart (a chain of them would wait for each other)
          if constexpr (kParts == 3) {
            // a step's are added up on their own, the small ones first: one rounding of the long sum per step
            f32x4_t sum[FN];
#pragma unroll
            for (int t = 0; t < kSplitProducts; ++t)
#pragma unroll
              for (int f = 0; f < FN; ++f)
                sum[f] = wgrad_mfma(fa[f][kSplitA[t]], fb[kSplitB[t]], t == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : sum[f]);
#pragma unroll
            for (int f = 0; f < FN; ++f) acc[f][g] += sum[f];
          } else {
#pragma unroll
            for (int f = 0; f < FN; ++f) acc[f][g] = wgrad_mfma(fa[f][0], fb[0], acc[f][g]);
          }
        }
      }
    }
  }
  float* part = job.part + static_cast<int64_t>(split) * job.stride;
  if (bias) {   // block-uniform
    __syncthreads();
    if (threadIdx.x < kTileN && n0 + threadIdx.x < job.n) {
      float v = 0.f;
#pragma unroll
      for (int g = 0; g < kGroups; ++g) v += s_sum[g][threadIdx.x];
      part[job.n * job.k + n0 + threadIdx.x] = v;
    }
  }
  if (!active) return;
  if constexpr (kParts == 3) {
    bool finite = true;
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
      for (int g = 0; g < FK; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) finite &= __builtin_isfinite(acc[f][g][q]);
    if (__any(!finite)) {   // again with the fp32 instruction, four rows at a time
#pragma unroll
      for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int g = 0; g < FK; ++g) acc[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int64_t r = group; r < m1 - m0 + group; r += 4) {
        float av[FN], bv[FK];
#pragma unroll
        for (int f = 0; f < FN; ++f) {
          const uint32_t at = static_cast<uint32_t>((r * job.n + wave_n + f * 16 + col16) * 4);
          av[f] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(dy, at, 0, 0));
          if (masked && __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(out, at, 0, 0)) <= 0.f) av[f] = 0.f;
        }
#pragma unroll
        for (int g = 0; g < FK; ++g)
          bv[g] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              x, static_cast<uint32_t>((r * job.k + wave_k + g * 16 + col16) * 4), 0, 0));
#pragma unroll
        for (int f = 0; f < FN; ++f)
#pragma unroll
          for (int g = 0; g < FK; ++g) acc[f][g] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[f], bv[g], acc[f][g], 0, 0, 0);
      }
    }
  }
  // Element q of a lane's accumulator is row (dy column) group * 4 + q, column (x column) lane % 16 of the fragment.
#pragma unroll
  for (int f = 0; f < FN; ++f)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t n = wave_n + f * 16 + wgrad_col<T>(group * 4 + q);
      if (n >= job.n) continue;
#pragma unroll
      for (int g = 0; g < FK; ++g) {
        const int64_t k = wave_k + g * 16 + col16;
        if (k < job.k) part[n * job.k + k] = acc[f][g][q];
      }
    }
}

// Sums of the partials of all products, in the order of the splits: 256 elements per workgroup, four per lane, the splits
// dealt to its wavefronts.
constexpr int kWgradSumBlock = 512;
constexpr int kWgradSumWaves = kWgradSumBlock / kWave;

template <typename E>
__global__ __launch_bounds__(kWgradSumBlock) void wgrad_sums_kernel(WgradParams p, int blocks0) {
  constexpr int kUnroll = 8;
  __shared__ __align__(16) f32x4_t s_sum[kWgradSumWaves][kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int which = static_cast<int>(blockIdx.x) >= blocks0 ? 1 : 0;
  const WgradJob& job = p.job[which];
  const int64_t e = (static_cast<int64_t>(blockIdx.x) - (which ? blocks0 : 0)) * (4 * kWave) + lane * 4;
  const bool live = e < job.stride;                     // (a multiple of four)
  const f32x4_t* src = reinterpret_cast<const f32x4_t*>(job.part + (live ? e : 0));
  const int64_t step = job.stride / 4;
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
  for (int s = wave; s < job.splits; s += kWgradSumWaves * kUnroll) {
    f32x4_t v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] = src[min(s + u * kWgradSumWaves, job.splits - 1) * step];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      if (s + u * kWgradSumWaves < job.splits) sum += v[u];
  }
  s_sum[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || !live) return;
#pragma unroll
  for (int w = 1; w < kWgradSumWaves; ++w) sum += s_sum[w][lane];
  const int64_t nk = job.n * job.k;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (e + q < nk) {
      if (job.dw != nullptr) static_cast<E*>(job.dw)[e + q] = from_float<E>(sum[q]);
    } else if (e + q < nk + job.n) {
      if (job.db != nullptr) static_cast<E*>(job.db)[e + q - nk] = from_float<E>(sum[q]);
    }
  }
}

static bool wgrad_sizes_ok(int64_t m, int64_t n, int64_t k) {
  return m >= 0 && n > 0 && k >= 0 && n <= (1 << 20) && k <= (1 << 20) && n * k <= (int64_t{1} << 30);
}

// Tiles of 128 x 128 where both sides of a product are longer than 64 and its rows make a workgroup for every CU, of
// 64 x 64 otherwise (the tile of 128 with half of it empty: 20 against 12 us for 10 k rows of 47 x 256 fp32).  The rows are
// split into as many parts as keep the CUs busy, while a part keeps two steps of its loop and the partials (written once,
// read once) stay below half of the inputs they come from or a few megabytes.  Both launches; before: a wavefront for
// itself loaded, regrouped and (fp32) split its operands, every tile's again.  us:
//   rows n x k            fp32 before / now      bf16 before / now
//   460 k 256 x 128           228 / 209              113 /  81
//   124 k 256 x 128            66 /  60               36 /  29
//   54 k  256 x 100            38 /  33               25 /  20
//   54 k  256 x (100 + 100)    87 /  60               53 /  26      (two products in one launch)
//   11 k  256 x (256 + 256)    77 /  34               52 /  22
//   20 k   47 x 256            24 /  16               21 /  11
//   20 k  256 x 602            62 /  52               37 /  26
//   20 k 1024 x 1024          274 / 247              123 /  87
//   460 k  47 x 256           135 / 142               70 /  63
//   460 k 256 x 64            139 / 150               76 /  60
//   460 k 512 x 64            248 / 272              129 / 117
//   460 k  41 x 602           365 / 312              209 / 149
// Where one side is at most 64 wide, the small tiles split an fp32 operand's rows for each of the tiles beside it.  Over long
// blocks that costs more than what an oblong tile's wavefronts lose by unequal shares.  fp32, 64 x 64 / oblong, us (m: masked):
//   60 k  47 x 256   28 /  30      124 k 512 x 64   85 /  84      300 k 256 x 64 m   152 / 140
//   60 k 512 x 64    44 /  47      124 k  41 x 602  98 /  92      460 k  47 x 256 m  198 / 164
//   124 k 256 x 64   44 /  46      460 k  47 x 256 153 / 142      460 k  41 x 602 m  657 / 360
//   460 k 128 x 64   91 /  91      460 k 512 x 64  284 / 272      (one tile: nothing to gain)
// bf16 has no split to save: 460 k rows of 256 x 64 61 / 67, of 128 x 64 35 / 39.
struct WgradSides { int n, k; };   // of a tile

static WgradSides wgrad_shape(WgradParams& p, int elem_size) {
  const int64_t step = elem_size == 4 ? 32 : 64;
  bool big = false, tall = elem_size == 4, wide = tall, is_long = false;
  for (int j = 0; j < p.jobs; ++j) {
    const WgradJob& w = p.job[j];
    big |= w.n > 64 && w.k > 64 && ceil_div(w.n, 128) * ceil_div(w.k, 128) * ceil_div(w.m, 2 * step) >= 256;
    if (w.k == 0) continue;
    tall &= w.n > 64 && w.k <= 64;
    wide &= w.n <= 64 && w.k > 64;
    is_long |= w.m * (ceil_div(w.n, 128) * ceil_div(w.k, 128)) >= kWgradLongRows;
  }
  tall &= is_long;
  wide &= is_long && !tall;
  const int64_t tile_n = big || tall ? 128 : 64, tile_k = big || wide ? 128 : 64;
  int64_t work = 0, part_row = 0, bytes = 0, most = 1, widest = 1;
  p.tiles = 0;
  for (int j = 0; j < p.jobs; ++j) {
    WgradJob& w = p.job[j];
    w.tiles_k = static_cast<int>(std::max<int64_t>(ceil_div(w.k, tile_k), 1));
    w.tiles = static_cast<int>(ceil_div(w.n, tile_n) * w.tiles_k);
    w.stride = ceil_div(w.n * w.k + w.n, 4) * 4;
    p.tiles += w.tiles;
    work += w.m * w.tiles;
    part_row += w.m * w.stride * 4;
    bytes += w.m * (w.n + w.k) * elem_size;
    most = std::max(most, w.m);
    widest = std::max(widest, std::max(w.n, w.k) * elem_size);
  }
  // rows of a split: from the workgroups aimed at, and from the partials' bytes (part_row / rows)
  int64_t rows = std::max(ceil_div(work, kWgradGroups), 2 * step);
  if (!big) rows = std::max({ceil_div(work, kWgradSmallGroups), std::min(rows, kWgradSmallSteps * step), 2 * step});
  rows = std::max(rows, ceil_div(part_row, std::max(kWgradPartBytes, bytes / 2)));
  rows = std::min(ceil_div(rows, step) * step, ceil_div(most, step) * step);
  // a split's rows are addressed with 32-bit offsets, and the loop reads up to 2 kWgradAhead steps past its last one
  const int64_t limit = std::max<int64_t>((int64_t{1} << 30) / widest / step, 1) * step;
  rows = std::min(rows, limit);
  // ... nor more workgroups than the CUs hold at a time: a few too many are a second round (300 k + 150 k masked rows of
  // 256 x 64: 236 us with 514 of them, 174 with 512)
  const auto groups = [&](int64_t r) {
    int64_t sum = 0;
    for (int j = 0; j < p.jobs; ++j) sum += ceil_div(p.job[j].m, r) * p.job[j].tiles;
    return sum;
  };
  const int64_t held = big ? kWgradGroups : kWgradSmallGroups;
  while (p.tiles <= held && rows < most && groups(rows) > held && rows < limit)
    rows = std::min(rows + ceil_div(rows, 64 * step) * step, limit);
  p.rows_per_split = rows;
  for (int j = 0; j < p.jobs; ++j) p.job[j].splits = static_cast<int>(ceil_div(p.job[j].m, rows));
  p.longer = p.jobs > 1 && p.job[1].splits > p.job[0].splits ? 1 : 0;
  p.common = p.jobs > 1 ? std::min(p.job[0].splits, p.job[1].splits) : p.job[0].splits;
  p.groups = static_cast<int>(groups(rows));
  return {static_cast<int>(tile_n), static_cast<int>(tile_k)};
}

static size_t wgrad_bytes(const WgradParams& p) {
  size_t bytes = 0;
  for (int j = 0; j < p.jobs; ++j) bytes += static_cast<size_t>(std::max(p.job[j].splits, 1)) * p.job[j].stride * sizeof(float);
  return bytes;
}

// Whether rows of bf16 can be read in pairs of columns.
static bool wgrad_pairs(const void* p, int64_t cols) { return cols % 2 == 0 && (reinterpret_cast<uintptr_t>(p) & 3) == 0; }

template <typename T>
static void launch_wgrad(const WgradParams& p, WgradSides tile, hipStream_t st) {
  const bool masked = p.job[0].out != nullptr || p.job[1].out != nullptr;
  const dim3 grid(static_cast<unsigned>(ceil_div(p.groups, 8) * 8)), block(kWgradBlock);
#define APT_WGRAD(N, K) \
  hipLaunchKernelGGL((masked ? wgrad_kernel<WgradRelu<T>, N, K> : wgrad_kernel<T, N, K>), grid, block, \
                     (WgradTile<T, N, K>::kLds), st, p)
  if (tile.n == 128 && tile.k == 128) {
    APT_WGRAD(4, 4);
  } else if (tile.n == tile.k) {
    APT_WGRAD(2, 2);
  } else if constexpr (WgradType<T>::kParts == 3) {
    if (tile.n > tile.k) APT_WGRAD(4, 2);
    else APT_WGRAD(2, 4);
  }
#undef APT_WGRAD
}

static int wgrad_params(const char* who, const apt_wgrad_product* products, int count, int elem_size, WgradParams& p) {
  APT_REQUIRE(products != nullptr && count >= 1 && count <= kWgradJobs, APT_EINVAL, "%s: %d products", who, count);
  APT_REQUIRE(elem_size == 2 || elem_size == 4, APT_EINVAL, "%s: elem_size %d (4 = fp32, 2 = bf16)", who, elem_size);
  p.jobs = count;
  for (int j = 0; j < count; ++j) {
    const apt_wgrad_product& q = products[j];
    APT_REQUIRE(wgrad_sizes_ok(q.m, q.n, q.k), APT_ELIMIT, "%s: sizes out of range (m %lld, n %lld, k %lld)", who,
                (long long)q.m, (long long)q.n, (long long)q.k);
    WgradJob& w = p.job[j];
    w.dy = q.dy;
    w.out = q.out;
    w.x = q.x;
    w.m = q.m;
    w.n = q.n;
    w.k = q.k;
    w.dw = q.dw;
    w.db = q.db;
  }
  return APT_OK;
}

}  // namespace apt

extern "C" size_t apt_linear_wgrads_workspace_bytes(const apt_wgrad_product* products, int count, int elem_size) {
  using namespace apt;
  WgradParams p{};
  if (wgrad_params("apt_linear_wgrads_workspace_bytes", products, count, elem_size, p) != APT_OK) return 0;
  wgrad_shape(p, elem_size);
  return wgrad_bytes(p);
}

extern "C" int apt_linear_wgrads(const apt_wgrad_product* products, int count, int elem_size, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  using namespace apt;
  const char* who = "apt_linear_wgrads";
  WgradParams p{};
  if (const int rc = wgrad_params(who, products, count, elem_size, p)) return rc;
  const WgradSides tile = wgrad_shape(p, elem_size);
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= wgrad_bytes(p) && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
              APT_EWORKSPACE, "%s: workspace too small or not 16-byte aligned (see apt_linear_wgrads_workspace_bytes)", who);
  float* part = static_cast<float*>(workspace);
  bool odd = false, any = false;
  int64_t sum_blocks[kWgradJobs] = {};
  for (int j = 0; j < p.jobs; ++j) {
    WgradJob& w = p.job[j];
    APT_REQUIRE((w.k == 0 || w.dw != nullptr) && (w.k > 0 || w.db != nullptr) &&
                    (w.m == 0 || (w.dy != nullptr && (w.k == 0 || w.x != nullptr))),
                APT_EINVAL, "%s: a tensor is NULL", who);
    w.part = part;
    part += static_cast<int64_t>(std::max(w.splits, 1)) * w.stride;
    odd |= !wgrad_pairs(w.dy, w.n) || !wgrad_pairs(w.out, w.n) || (w.k > 0 && !wgrad_pairs(w.x, w.k));
    any |= w.splits > 0;
    sum_blocks[j] = ceil_div(w.stride, 4 * kWave);   // (no rows: zeros)
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (any) {
    if (elem_size == 4) launch_wgrad<float>(p, tile, st);
    else if (odd) launch_wgrad<WgradOdd>(p, tile, st);
    else launch_wgrad<uint16_t>(p, tile, st);
    APT_LAUNCH_CHECK("wgrad_kernel");
  }
  const dim3 grid(static_cast<unsigned>(sum_blocks[0] + sum_blocks[1])), block(kWgradSumBlock);
  const int blocks0 = static_cast<int>(sum_blocks[0]);
  if (elem_size == 4) hipLaunchKernelGGL(wgrad_sums_kernel<float>, grid, block, 0, st, p, blocks0);
  else hipLaunchKernelGGL(wgrad_sums_kernel<uint16_t>, grid, block, 0, st, p, blocks0);
  APT_LAUNCH_CHECK("wgrad_sums_kernel");
  return APT_OK;
}

extern "C" size_t apt_linear_wgrad_workspace_bytes(int64_t m, int64_t n, int64_t k, int elem_size) {
  if (k < 1) return 0;
  const apt_wgrad_product q{nullptr, nullptr, nullptr, m, n, k, nullptr, nullptr};
  return apt_linear_wgrads_workspace_bytes(&q, 1, elem_size);
}

extern "C" int apt_linear_wgrad(const void* dy, const void* x, int64_t m, int64_t n, int64_t k, int elem_size, void* dw,
                                void* db, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(k > 0, APT_ELIMIT, "apt_linear_wgrad: sizes out of range (m %lld, n %lld, k %lld)", (long long)m, (long long)n,
              (long long)k);
  const apt_wgrad_product q{dy, nullptr, x, m, n, k, dw, db};
  return apt_linear_wgrads(&q, 1, elem_size, workspace, workspace_bytes, stream);
}

// Gradients of a dense layer's weight and bias over the rows of a block:
//   dw[n, k] = sum_m dy[m, n] * x[m, k],   db[n] = sum_m dy[m, n]
//
// A block has 10^4..10^6 rows and a layer a few hundred columns, so this product
// reduces over the one long dimension and its output is a few tiles: bound by
// reading dy and x once (bf16) or by the fp32 matrix rate.  A GEMM that gives
// every output tile to one workgroup keeps a handful of the 256 CUs busy; here
// the rows are split over the chip, every workgroup accumulates the whole output
// of its rows in MFMA accumulators and leaves it in a partial buffer, and a second
// launch adds the partials in a fixed order (reproducible, no atomics).
//
// fp32 operands are multiplied as bf16 parts (split_bf16.hpp): the fp32 matrix
// instruction would bound the product (57 us of its rate alone for 71 k rows of
// 256 x 100 in tiles of 64; the four 256-wide gradients of a GraphSAGE step of
// 4096 seeds took 169 us with it and take 132).
// Both operands have the reduced dimension as their row index, which is what an
// MFMA operand wants *inside* a lane (8 consecutive rows of one column).  No LDS transpose: a lane loads VEC consecutive columns of each
// of its rows and the 16-bit halves are regrouped by column in registers
// (v_perm); the columns of the MFMA tiles are simply numbered lane * VEC + j.
#include <algorithm>

#include "common.hpp"
#include "partial_sums.hpp"
#include "split_bf16.hpp"

namespace apt {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// Buffer loads: a range-checked base in scalar registers plus a 32-bit lane offset; what lies past the range reads
// as zero, so neither the last rows of a split nor the columns past the edge of a tile need a branch.
typedef uint32_t u32x2_v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_v __attribute__((ext_vector_type(4)));
using buffer_t = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ buffer_t make_buffer(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<uint32_t>(bytes), 0x00020000);
}

constexpr int kWgradTile = 64;      // output columns of dy / of x per wavefront
constexpr int kWgradFrags = kWgradTile / 16;
constexpr int kWgradWaves = 8;
constexpr int kWgradGroups = 256;                     // workgroups aimed at: one per CU
constexpr int64_t kWgradMinRows = 64;                 // rows a split has at least
constexpr int64_t kWgradPartBytes = int64_t{12} << 20;

struct WgradParams {
  const void* dy;      // [m, n]
  const void* x;       // [m, k]
  int64_t m, n, k;
  float* part;         // [splits][n * k + n]
  int64_t part_stride;
  int tiles_k, tiles;  // wavefront tiles of the output (tiles_n * tiles_k)
  int tile_groups;     // workgroups per split: ceil(tiles / waves)
  int splits_per_group;  // splits in a workgroup where tile_groups == 1
  int splits;
  int64_t rows_per_split;
};

constexpr int kWgradRows = 32;     // rows per step: one MFMA of depth 32 (fp32: six, of its bf16 parts)
constexpr int kWgradLoads = 8;     // consecutive rows of a lane in a step; the lanes of a 16-lane group share them

// The lane's rows of one operand as they come from memory: VEC consecutive columns of each row (VEC 4), two pairs
// (VEC 2) or kWgradFrags single columns (VEC 1), at the byte offsets off[].  What an MFMA wants is taken out of it
// only when it is used: regrouping at the load would wait for it.
template <typename T, int VEC> struct WgradRows {
  static constexpr int kWords = sizeof(T) == 4 || VEC == 1 ? kWgradFrags : 2;   // 32-bit registers per row
  static constexpr int kOffsets = kWgradFrags / VEC;
  uint32_t v[kWgradLoads][kWords];
  __device__ __forceinline__ void load(buffer_t buf, uint32_t at, uint32_t row_bytes, const uint32_t (&off)[kOffsets]) {
#pragma unroll
    for (int r = 0; r < kWgradLoads; ++r, at += row_bytes) {
      if constexpr (VEC * sizeof(T) == 16) {
        const u32x4_v w = __builtin_amdgcn_raw_buffer_load_b128(buf, off[0] + at, 0, 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) v[r][c] = w[c];
      } else if constexpr (VEC * sizeof(T) == 8) {
#pragma unroll
        for (int o = 0; o < kOffsets; ++o) {
          const u32x2_v w = __builtin_amdgcn_raw_buffer_load_b64(buf, off[o] + at, 0, 0);
          v[r][2 * o] = w[0];
          v[r][2 * o + 1] = w[1];
        }
      } else {
#pragma unroll
        for (int o = 0; o < kOffsets; ++o) {
          if constexpr (VEC * sizeof(T) == 4) v[r][o] = __builtin_amdgcn_raw_buffer_load_b32(buf, off[o] + at, 0, 0);
          else v[r][o] = __builtin_amdgcn_raw_buffer_load_b16(buf, off[o] + at, 0, 0);
        }
      }
    }
  }
};

// Column of the output that element i (0..15) of tile fragment f stands for, relative to the tile.
template <int VEC>
__device__ __forceinline__ int wgrad_col(int f, int i) {
  return VEC == 4 ? i * 4 + f : VEC == 2 ? (f / 2) * 32 + i * 2 + (f & 1) : f * 16 + i;
}

// MFMA operands of one step: fragment f = 16 columns, the lane's rows of one of them.
template <typename T> struct WgradOperand;
template <> struct WgradOperand<float> {
  uint32_t v[3][kWgradFrags][4];   // the parts of eight values of a column, two rows to a register
  template <int VEC> __device__ __forceinline__ explicit WgradOperand(const WgradRows<float, VEC>& rows) {
#pragma unroll
    for (int f = 0; f < kWgradFrags; ++f)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const SplitPair s = split_pair(__uint_as_float(rows.v[2 * d][f]), __uint_as_float(rows.v[2 * d + 1][f]));
        v[0][f][d] = s.hi;
        v[1][f][d] = s.mid;
        v[2][f][d] = s.lo;
      }
  }
};
template <> struct WgradOperand<uint16_t> {
  uint32_t v[kWgradFrags][4];   // eight bf16 of a column, two rows to a register
  template <int VEC> __device__ __forceinline__ explicit WgradOperand(const WgradRows<uint16_t, VEC>& rows) {
#pragma unroll
    for (int f = 0; f < kWgradFrags; ++f)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int w = VEC == 1 ? f : f / 2;
        v[f][d] = __builtin_amdgcn_perm(rows.v[2 * d + 1][w], rows.v[2 * d][w],
                                        VEC != 1 && (f & 1) != 0 ? 0x07060302u : 0x05040100u);
      }
  }
};

// acc[fa][fb] += a[fa]^T b[fb] over the step's rows; products of one accumulator are kept apart (a chain of them
// would wait for each other).
__device__ __forceinline__ f32x4_t wgrad_mfma(const uint32_t (&a)[4], const uint32_t (&b)[4], f32x4_t acc) {
  const u32x4_v av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), __builtin_bit_cast(bf16x8_t, bv), acc,
                                                 0, 0, 0);
}
__device__ __forceinline__ void wgrad_products(const WgradOperand<float>& a, const WgradOperand<float>& b,
                                               f32x4_t (&acc)[kWgradFrags][kWgradFrags]) {
#pragma unroll
  for (int t = 0; t < kSplitProducts; ++t)
#pragma unroll
    for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
      for (int fb = 0; fb < kWgradFrags; ++fb)
        acc[fa][fb] = wgrad_mfma(a.v[kSplitA[t]][fa], b.v[kSplitB[t]][fb], acc[fa][fb]);
}
__device__ __forceinline__ void wgrad_products(const WgradOperand<uint16_t>& a, const WgradOperand<uint16_t>& b,
                                               f32x4_t (&acc)[kWgradFrags][kWgradFrags]) {
#pragma unroll
  for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
    for (int fb = 0; fb < kWgradFrags; ++fb) acc[fa][fb] = wgrad_mfma(a.v[fa], b.v[fb], acc[fa][fb]);
}
// Column sums of dy.  bf16: a product with ones (4 more MFMAs beside 16; unpacking the halves would cost more), the
// sum of column i in accumulator row i.  fp32: the vector units add; the lane's sum covers its own rows of columns l16.
template <int VEC>
__device__ __forceinline__ void wgrad_sums(const WgradRows<uint16_t, VEC>&, const WgradOperand<uint16_t>& a,
                                           f32x4_t (&sum)[kWgradFrags]) {
  const uint32_t ones[4] = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
#pragma unroll
  for (int f = 0; f < kWgradFrags; ++f) sum[f] = wgrad_mfma(a.v[f], ones, sum[f]);
}
template <int VEC>
__device__ __forceinline__ void wgrad_sums(const WgradRows<float, VEC>& rows, const WgradOperand<float>&,
                                           f32x4_t (&sum)[kWgradFrags]) {
#pragma unroll
  for (int f = 0; f < kWgradFrags; ++f)
#pragma unroll
    for (int r = 0; r < kWgradLoads; ++r) sum[f][r & 1] += __uint_as_float(rows.v[r][f]);
}

template <typename T, int VA, int VB>
__global__ __launch_bounds__(kWgradWaves * kWave) void wgrad_kernel(WgradParams p) {
  constexpr int kRows = kWgradRows;
  const int lane = threadIdx.x % kWave;
  const int l16 = lane % 16, group = lane / 16;
  // A wavefront has one tile of one split.  The workgroups of a split read the same rows: they are numbered eight
  // apart, i.e. on one XCD, whose L2 then serves the second reader.
  int split, tile;
  const int wave = threadIdx.x / kWave;
  if (p.tile_groups == 1) {
    split = blockIdx.x * p.splits_per_group + wave / p.tiles;
    tile = wave % p.tiles;
    if (wave >= p.splits_per_group * p.tiles) return;
  } else {
    const int i = blockIdx.x / 8;
    split = (i / p.tile_groups) * 8 + blockIdx.x % 8;
    tile = (i % p.tile_groups) * kWgradWaves + wave;
  }
  split = __builtin_amdgcn_readfirstlane(split);
  tile = __builtin_amdgcn_readfirstlane(tile);
  if (split >= p.splits || tile >= p.tiles) return;   // wave-uniform, no barriers below
  const int64_t n0 = static_cast<int64_t>(tile / p.tiles_k) * kWgradTile;
  const int64_t k0 = static_cast<int64_t>(tile % p.tiles_k) * kWgradTile;
  const int64_t m0 = static_cast<int64_t>(split) * p.rows_per_split;
  const int64_t m1 = min(m0 + p.rows_per_split, p.m);
  const buffer_t dy = make_buffer(static_cast<const T*>(p.dy) + m0 * p.n, (m1 - m0) * p.n * sizeof(T));
  const buffer_t x = make_buffer(static_cast<const T*>(p.x) + m0 * p.k, (m1 - m0) * p.k * sizeof(T));
  // A lane's offsets inside a step do not change.  Columns past the edge read the row after (or zero): they only
  // reach outputs past the edge, which are not stored.
  uint32_t off_a[kWgradFrags / VA], off_b[kWgradFrags / VB];
#pragma unroll
  for (int o = 0; o < kWgradFrags / VA; ++o)
    off_a[o] = static_cast<uint32_t>((group * kWgradLoads * p.n + n0 + wgrad_col<VA>(o * VA, l16)) * sizeof(T));
#pragma unroll
  for (int o = 0; o < kWgradFrags / VB; ++o)
    off_b[o] = static_cast<uint32_t>((group * kWgradLoads * p.k + k0 + wgrad_col<VB>(o * VB, l16)) * sizeof(T));
  const uint32_t row_a = static_cast<uint32_t>(p.n * sizeof(T)), row_b = static_cast<uint32_t>(p.k * sizeof(T));
  const uint32_t step_a = static_cast<uint32_t>(kRows * p.n * sizeof(T)), step_b = static_cast<uint32_t>(kRows * p.k * sizeof(T));
  f32x4_t acc[kWgradFrags][kWgradFrags] = {};
  f32x4_t sum[kWgradFrags] = {};
  const bool bias = tile % p.tiles_k == 0;

  const int steps = static_cast<int>((m1 - m0 + kRows - 1) / kRows);
  uint32_t at_a = 0, at_b = 0;
  WgradRows<T, VA> a0;
  WgradRows<T, VB> b0;
  a0.load(dy, at_a, row_a, off_a);
  b0.load(x, at_b, row_b, off_b);
  if constexpr (sizeof(T) == 4) {
    // The parts take the place of the second step's rows (registers): the next rows are on their way during the products.
    for (int s = 0; s < steps; ++s) {
      const WgradOperand<T> oa(a0), ob(b0);
      if (bias) wgrad_sums(a0, oa, sum);
      at_a += step_a;
      at_b += step_b;
      a0.load(dy, at_a, row_a, off_a);
      b0.load(x, at_b, row_b, off_b);
      wgrad_products(oa, ob, acc);
    }
    bool finite = true;
#pragma unroll
    for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
      for (int fb = 0; fb < kWgradFrags; ++fb)
#pragma unroll
        for (int q = 0; q < 4; ++q) finite &= __builtin_isfinite(acc[fa][fb][q]);
    if (__any(!finite)) {   // again with the fp32 instruction (rows r, 8 + r, 16 + r, 24 + r of a step at a time)
#pragma unroll
      for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
        for (int fb = 0; fb < kWgradFrags; ++fb) acc[fa][fb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      at_a = at_b = 0;
#pragma unroll 1
      for (int s = 0; s < steps; ++s, at_a += step_a, at_b += step_b) {
        a0.load(dy, at_a, row_a, off_a);
        b0.load(x, at_b, row_b, off_b);
#pragma unroll
        for (int r = 0; r < kWgradLoads; ++r)
#pragma unroll
          for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
            for (int fb = 0; fb < kWgradFrags; ++fb)
              acc[fa][fb] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a0.v[r][fa]), __uint_as_float(b0.v[r][fb]),
                                                                 acc[fa][fb], 0, 0, 0);
      }
    }
  } else {
    auto multiply = [&](const WgradRows<T, VA>& a, const WgradRows<T, VB>& b) {
      const WgradOperand<T> oa(a), ob(b);
      wgrad_products(oa, ob, acc);
      if (bias) wgrad_sums(a, oa, sum);
    };
    // Two steps in registers: the rows of one are on their way during the products of the other.  A step past the
    // split's end reads zeros.
    WgradRows<T, VA> a1;
    WgradRows<T, VB> b1;
    for (int s = 0; s < steps; s += 2) {
      at_a += step_a;
      at_b += step_b;
      a1.load(dy, at_a, row_a, off_a);
      b1.load(x, at_b, row_b, off_b);
      multiply(a0, b0);
      at_a += step_a;
      at_b += step_b;
      a0.load(dy, at_a, row_a, off_a);
      b0.load(x, at_b, row_b, off_b);
      multiply(a1, b1);
    }
  }
  // Element q of a lane's accumulator is row (dy column) group * 4 + q, column (x column) l16 of the tile fragment.
  float* part = p.part + static_cast<int64_t>(split) * p.part_stride;
#pragma unroll
  for (int fa = 0; fa < kWgradFrags; ++fa)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t n = n0 + wgrad_col<VA>(fa, group * 4 + q);
      if (n >= p.n) continue;
#pragma unroll
      for (int fb = 0; fb < kWgradFrags; ++fb) {
        const int64_t k = k0 + wgrad_col<VB>(fb, l16);
        if (k < p.k) part[n * p.k + k] = acc[fa][fb][q];
      }
      if (sizeof(T) == 2 && bias && l16 == 0) part[p.n * p.k + n] = sum[fa][q];
    }
  if (sizeof(T) == 4 && bias) {
#pragma unroll
    for (int f = 0; f < kWgradFrags; ++f) {
      float v = sum[f][0] + sum[f][1];
      v += __shfl_xor(v, 16, kWave);
      v += __shfl_xor(v, 32, kWave);
      const int64_t n = n0 + wgrad_col<VA>(f, l16);
      if (group == 0 && n < p.n) part[p.n * p.k + n] = v;
    }
  }
}

// How the rows are split: into as many parts as keep eight wavefronts on every CU, while a part keeps a few steps of
// its loop and the partials (written once, read once) stay below half of the inputs they come from or a few
// megabytes.  Both launches, against the library's GEMM and column sum, for n x k = 256 x 128:
//   rows      bf16: here / library     fp32: here / library
//   256              18 / 27 us              20 / 42 us
//   17 k             25 / 108 us             33 / 120 us     (fp32 instruction:  40)
//   170 k            46 / 403 us            101 / 358 us     (118; bytes alone 52, products 66 at the bf16 rate)
//   700 k           171 / 1435 us           436 / 1385 us    (431)
static void wgrad_shape(int64_t m, int64_t n, int64_t k, int elem_size, WgradParams& p) {
  const int64_t tiles_n = ceil_div(n, kWgradTile);
  p.tiles_k = static_cast<int>(ceil_div(k, kWgradTile));
  p.tiles = static_cast<int>(tiles_n * p.tiles_k);
  p.tile_groups = static_cast<int>(ceil_div(p.tiles, kWgradWaves));
  p.splits_per_group = p.tile_groups == 1 ? kWgradWaves / p.tiles : 1;
  p.part_stride = n * k + n;
  const int64_t part_bytes = p.part_stride * 4;
  int64_t s = p.tile_groups == 1 ? kWgradGroups * p.splits_per_group : ceil_div(kWgradGroups, p.tile_groups);
  s = std::min(s, std::max(kWgradPartBytes, m * (n + k) * elem_size / 2) / part_bytes);
  s = std::max<int64_t>(1, std::min(s, ceil_div(m, kWgradMinRows)));
  // a split's rows are addressed with 32-bit offsets, and the loop reads up to three steps past its last one
  s = std::max(s, ceil_div(m * std::max(n, k) * elem_size, int64_t{1} << 30));
  p.rows_per_split = ceil_div(ceil_div(m, s), kWgradRows) * kWgradRows;
  p.splits = static_cast<int>(ceil_div(m, p.rows_per_split));
}

template <typename T>
static void launch_wgrad(const WgradParams& p, int va, int vb, hipStream_t st) {
  const int64_t groups = p.tile_groups == 1 ? ceil_div(p.splits, p.splits_per_group)
                                            : ceil_div(p.splits, 8) * 8 * p.tile_groups;
  const dim3 grid(static_cast<unsigned>(groups)), block(kWgradWaves * kWave);
#define APT_WGRAD(VA, VB) hipLaunchKernelGGL((wgrad_kernel<T, VA, VB>), grid, block, 0, st, p)
#define APT_WGRAD_B(VA)              \
  if (vb == 4) APT_WGRAD(VA, 4);     \
  else if (vb == 2) APT_WGRAD(VA, 2); \
  else APT_WGRAD(VA, 1)
  if (va == 4) { APT_WGRAD_B(4); }
  else if (va == 2) { APT_WGRAD_B(2); }
  else { APT_WGRAD_B(1); }
#undef APT_WGRAD_B
#undef APT_WGRAD
}

static int wgrad_vec(const void* p, int64_t cols, int elem_size) {
  for (int v = 4; v > 1; v >>= 1)
    if (cols % v == 0 && (reinterpret_cast<uintptr_t>(p) & (v * elem_size - 1)) == 0) return v;
  return 1;
}

static bool wgrad_sizes_ok(int64_t m, int64_t n, int64_t k) {
  return m >= 0 && n > 0 && k > 0 && n <= (1 << 20) && k <= (1 << 20) && n * k <= (int64_t{1} << 30);
}

}  // namespace apt

extern "C" size_t apt_linear_wgrad_workspace_bytes(int64_t m, int64_t n, int64_t k, int elem_size) {
  using namespace apt;
  if (!wgrad_sizes_ok(m, n, k) || (elem_size != 2 && elem_size != 4)) return 0;
  WgradParams p{};
  wgrad_shape(std::max<int64_t>(m, 1), n, k, elem_size, p);
  return static_cast<size_t>(p.splits) * p.part_stride * sizeof(float);
}

extern "C" int apt_linear_wgrad(const void* dy, const void* x, int64_t m, int64_t n, int64_t k, int elem_size, void* dw,
                                void* db, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(wgrad_sizes_ok(m, n, k), APT_ELIMIT, "apt_linear_wgrad: sizes out of range (m %lld, n %lld, k %lld)",
              (long long)m, (long long)n, (long long)k);
  APT_REQUIRE(elem_size == 2 || elem_size == 4, APT_EINVAL, "apt_linear_wgrad: elem_size %d (4 = fp32, 2 = bf16)",
              elem_size);
  APT_REQUIRE(dw != nullptr && (m == 0 || (dy != nullptr && x != nullptr)), APT_EINVAL,
              "apt_linear_wgrad: a tensor is NULL");
  WgradParams p{};
  p.dy = dy;
  p.x = x;
  p.m = m;
  p.n = n;
  p.k = k;
  p.part = static_cast<float*>(workspace);
  wgrad_shape(std::max<int64_t>(m, 1), n, k, elem_size, p);
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= static_cast<size_t>(p.splits) * p.part_stride * sizeof(float) &&
                  (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
              APT_EWORKSPACE, "apt_linear_wgrad: workspace too small or not 16-byte aligned "
                              "(see apt_linear_wgrad_workspace_bytes)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (m == 0) p.splits = 0;   // the reduction then writes zeros
  if (p.splits > 0) {
    const int va = wgrad_vec(dy, n, elem_size), vb = wgrad_vec(x, k, elem_size);
    if (elem_size == 4) launch_wgrad<float>(p, va, vb, st);
    else launch_wgrad<uint16_t>(p, va, vb, st);
    APT_LAUNCH_CHECK("wgrad_kernel");
  }
  if (elem_size == 4) launch_partial_sums<float, float>(p.part, p.part_stride, p.splits, dw, n * k, db, n, nullptr, 0, st);
  else launch_partial_sums<uint16_t, uint16_t>(p.part, p.part_stride, p.splits, dw, n * k, db, n, nullptr, 0, st);
  APT_LAUNCH_CHECK("partial_sums_kernel");
  return APT_OK;
}

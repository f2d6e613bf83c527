// The dense product of a layer over a block's rows in bf16, two operand pairs at once:
//   y[r, :] = x1[r, :] w1^T + x2[r, :] w2^T + bias        (x2 for the first m2 rows only)
// with fp32 sums that are rounded once, where they are stored (the fp32 counterpart is rows_gemm.hip).
//
// Bound by reading the rows and writing the result: a layer has a few hundred columns, so its weights fit LDS.  A
// workgroup brings those of its column tile there once, in the order of the MFMA operand, and keeps them while its
// wavefronts walk over their share of the rows, sixteen at a time and all columns of the tile; the rows go from memory
// straight into operand registers, four steps of the product ahead, across the ends of the tiles.  The columns of a fragment
// pair are dealt to the lanes so that a lane has eight neighbouring results of a row: one 16-byte store.
//
// us, here / the library's GEMM (floor: rows and result at 5.7 TB/s):
//   124 k rows, 128 -> 256   23 / 44 (17)     460 k, 128 -> 64    31 / 57 (31)     460 k, 100 -> 256  101 / 172 (58)
//   19 k, 256 -> 256         13 / 13          3 k, 188 -> 256      7 / 8           rows of 200 bytes begin inside a line
//   54 k, 100 + 100 -> 256   23 / 48, with bias, ReLU and the sum of the two
// A workgroup's first rows wait for its weights (64 KB: 5 us), which is what small launches spend their time on.
#include <algorithm>

#include "common.hpp"
#include "feature_rows.hpp"

namespace apt {

typedef float prod_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t prod_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 prod_bf16x8 __attribute__((ext_vector_type(8)));
using prod_buffer_t = __amdgpu_buffer_rsrc_t;

constexpr int kProdWaves = 8;
constexpr int kProdBlock = kProdWaves * kWave;
constexpr int kProdStep = 32;              // depth of an MFMA
constexpr int kProdChunk = 4;              // steps whose rows are loaded together
constexpr int kProdFrags = 4;              // fragments of 64 columns
constexpr int kProdRows = kProdWaves * 16; // rows of a workgroup at once
constexpr int kProdLds = 128 << 10;        // bytes of weights at the most
constexpr int kProdGroups = 512;           // workgroups aimed at: two per CU

struct ProdOperand {
  const uint16_t* x;       // [rows, k]
  const uint16_t* w;       // [n, k] with these strides, one of which is 1
  int64_t rows;
  int k, steps;            // steps: of depth 32
  int64_t stride_n, stride_k;
};
struct ProdParams {
  ProdOperand a[2];
  int64_t m;
  int n, tiles_n, walkers;   // walkers: workgroups of a column tile
  int64_t row_blocks;
  const uint16_t* bias;
  int accumulate, relu, wide;   // wide: results that can be stored at a time
  uint16_t* y;
};

// Rows from a base on: a range-checked buffer (what lies past it reads as zero) that begins at a multiple of four bytes, and
// how far behind that the base is.  The last dword may hold half an element too many.
struct ProdRows {
  prod_buffer_t buffer;
  uint32_t skip;
  __device__ __forceinline__ ProdRows(const uint16_t* base, int64_t elems) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(base);
    skip = static_cast<uint32_t>(at & 3);
    const int64_t bytes = elems > 0 ? (elems * 2 + skip + 3) / 4 * 4 : 0;
    buffer = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at - skip), 0,
                                               static_cast<uint32_t>(min(bytes, static_cast<int64_t>(0x7ffffffc))), 0x00020000);
  }
};
// Eight elements from a byte offset on as they come from memory.  ODD: the offset need not be a multiple of four; a dword
// more is read, and value() takes the elements out of the five.
template <bool ODD> struct ProdRaw {
  prod_u32x4 v;
  uint32_t last;
  __device__ __forceinline__ void load(const ProdRows& rows, uint32_t at) {
    at += rows.skip;
    v = __builtin_bit_cast(prod_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rows.buffer, ODD ? at & ~3u : at, 0, 0));
    if constexpr (ODD) last = __builtin_amdgcn_raw_buffer_load_b32(rows.buffer, (at & ~3u) + 16, 0, 0);
  }
  __device__ __forceinline__ prod_u32x4 value(const ProdRows& rows, uint32_t at) const {
    if constexpr (!ODD) return v;
    const uint32_t shift = (at + rows.skip & 2) * 8;
    return prod_u32x4{__builtin_amdgcn_alignbit(v[1], v[0], shift), __builtin_amdgcn_alignbit(v[2], v[1], shift),
                      __builtin_amdgcn_alignbit(v[3], v[2], shift), __builtin_amdgcn_alignbit(last, v[3], shift)};
  }
};
// The first `count` of eight elements, zeros behind them.
__device__ __forceinline__ prod_u32x4 prod_first(prod_u32x4 v, int count) {
#pragma unroll
  for (int d = 0; d < 4; ++d) v[d] &= count >= 2 * d + 2 ? 0xffffffffu : count == 2 * d + 1 ? 0xffffu : 0u;
  return v;
}
// Fragment and element of column c (of 64) and the reverse (prod_column): lane group g has, of fragments 2 f and 2 f + 1,
// the columns 32 f + 8 g .. + 7.
__device__ __forceinline__ int prod_fragment(int c) { return c / 32 * 2 + c % 8 / 4; }
__device__ __forceinline__ int prod_element(int c) { return c % 32 / 8 * 4 + c % 4; }

// The weights of columns n0 .. n0 + 64 WN - 1 in LDS: [step][column fragment][lane].
template <int WN, bool ODD>
__device__ __forceinline__ void prod_stage_weights(const ProdOperand& a, int step0, int n, int n0, prod_u32x4* s_w) {
  constexpr int kCols = 64 * WN, kFragsN = kProdFrags * WN;
  const ProdRows rows(a.w, a.stride_k == 1 ? (static_cast<int64_t>(n) - 1) * a.stride_n + a.k
                                           : (static_cast<int64_t>(a.k) - 1) * a.stride_k + n);
  auto place = [&](int c, int kg, prod_u32x4 v) {   // kg: which eight of the depth
    s_w[((step0 + kg / 4) * kFragsN + c / 64 * kProdFrags + prod_fragment(c % 64)) * kWave + kg % 4 * 16 + prod_element(c % 64)] = v;
  };
  if (a.stride_k == 1) {      // a column's depth is contiguous
    constexpr int kBatch = 4;
    const int all = kCols * a.steps * 4;   // (neighbouring lanes have neighbouring columns: their stores to LDS do not collide)
    for (int i0 = threadIdx.x; i0 < all; i0 += kBatch * kProdBlock) {
      ProdRaw<ODD> v[kBatch];
      uint32_t at[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = min(i0 + u * kProdBlock, all - 1), c = i % kCols, kg = i / kCols;
        at[u] = static_cast<uint32_t>(((n0 + c) * a.stride_n + kg * 8) * 2);
        v[u].load(rows, at[u]);
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = i0 + u * kProdBlock, c = i % kCols, kg = i / kCols;
        if (i < all) place(c, kg, prod_first(v[u].value(rows, at[u]), a.k - kg * 8));
      }
    }
  } else {                    // the columns are: eight by eight elements, turned in registers
    constexpr int kPer = kCols / 8;
    const int all = kPer * a.steps * 4;
    for (int i = threadIdx.x; i < all; i += kProdBlock) {
      const int c = i % kPer * 8, kg = i / kPer;
      ProdRaw<ODD> raw[8];
      prod_u32x4 v[8];
      const uint32_t at = static_cast<uint32_t>((kg * 8 * a.stride_k + n0 + c) * 2), row = static_cast<uint32_t>(a.stride_k * 2);
#pragma unroll
      for (int r = 0; r < 8; ++r) raw[r].load(rows, at + r * row);
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = raw[r].value(rows, at + r * row);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        prod_u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          o[d] = __builtin_amdgcn_perm(v[2 * d + 1][q / 2], v[2 * d][q / 2], (q & 1) != 0 ? 0x07060302u : 0x05040100u);
        place(c + q, kg, prod_first(o, a.k - kg * 8));
      }
    }
  }
}

// WN: groups of 64 columns of the tile.
template <int WN, bool ODD>
__global__ __launch_bounds__(kProdBlock, 4) void rows_product_kernel(ProdParams p) {
  constexpr int kFragsN = kProdFrags * WN;
  extern __shared__ __align__(16) prod_u32x4 s_weights[];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l16 = lane % 16, group = lane / 16;
  // The workgroups of the same rows (other columns) follow each other on one XCD.
  const int i = static_cast<int>(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8);
  const int64_t first = __builtin_amdgcn_readfirstlane(i / p.tiles_n), stride = p.walkers;
  const int tile = __builtin_amdgcn_readfirstlane(i % p.tiles_n);
  if (first >= stride) return;   // block-uniform (the grid is a multiple of eight)
  const int n0 = tile * WN * 64;
  const int steps = p.a[0].steps + p.a[1].steps;
  float* s_bias = reinterpret_cast<float*>(s_weights + steps * kFragsN * kWave);
  prod_stage_weights<WN, ODD>(p.a[0], 0, p.n, n0, s_weights);
  if (p.a[1].steps > 0) prod_stage_weights<WN, ODD>(p.a[1], p.a[0].steps, p.n, n0, s_weights);
  for (int c = threadIdx.x; c < WN * 64; c += kProdBlock)
    s_bias[c] = p.bias != nullptr && n0 + c < p.n ? to_float<uint16_t>(p.bias[n0 + c]) : 0.f;
  __syncthreads();
  // (no barriers below)
  // The wavefront's work is a sequence of chunks of kProdChunk steps: of the first operand, then of the second, then of the
  // next tile of rows.
  struct At {
    int64_t block;     // of rows
    int which, step;
  };
  auto row0 = [&](const At& at) { return at.block * kProdRows + wave * 16; };
  auto next = [&](At at) {
    at.step += kProdChunk;
    if (at.step >= p.a[at.which].steps) {
      at.step = 0;
      if (at.which == 0 && p.a[1].steps > 0 && row0(at) < p.a[1].rows) {
        at.which = 1;
      } else {
        at.which = 0;
        at.block += stride;
      }
    }
    return at;
  };
  auto rows_of = [&](const At& at) {
    const ProdOperand& a = p.a[at.which];
    const int64_t row = min(row0(at), a.rows);   // (past the end: an empty range)
    return ProdRows(a.x + row * a.k, min(a.rows - row, static_cast<int64_t>(16)) * a.k);
  };
  auto offset = [&](const At& at, int s) {
    return static_cast<uint32_t>((l16 * p.a[at.which].k + (at.step + s) * kProdStep + group * 8) * 2);
  };
  ProdRaw<ODD> x[2][kProdChunk];
  auto load = [&](const At& at, ProdRaw<ODD> (&v)[kProdChunk]) {
    const ProdRows rows = rows_of(at);
#pragma unroll
    for (int s = 0; s < kProdChunk; ++s)   // (a step behind the last one: beyond the range, nothing is read)
      v[s].load(rows, offset(at, s) | (at.step + s < p.a[at.which].steps ? 0u : 0x80000000u));
  };
  prod_f32x4 acc[kFragsN];
  auto begin = [&]() {
#pragma unroll
    for (int f = 0; f < kFragsN; ++f)
      acc[f] = *reinterpret_cast<const prod_f32x4*>(s_bias + f / 2 * 32 + group * 8 + f % 2 * 4);
  };
  auto multiply = [&](const At& at, ProdRaw<ODD> (&v)[kProdChunk]) {
    const ProdOperand& a = p.a[at.which];
    const int base = at.which == 0 ? 0 : p.a[0].steps;
    const ProdRows rows = rows_of(at);
#pragma unroll
    for (int s = 0; s < kProdChunk; ++s) {
      if (at.step + s >= a.steps) continue;   // wave-uniform
      prod_u32x4 xs = v[s].value(rows, offset(at, s));
      const int left = a.k - (at.step + s) * kProdStep - group * 8;
      // The rows' last step reaches into the next row; ODD: the last row's last dword into what is no row at all.
      if constexpr (ODD) xs = prod_first(xs, row0(at) + l16 < a.rows ? left : 0);
      else if (at.step + s + 1 == a.steps) xs = prod_first(xs, left);
      const prod_u32x4* w = s_weights + (base + at.step + s) * kFragsN * kWave + lane;
#pragma unroll
      for (int f = 0; f < kFragsN; ++f)
        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(prod_bf16x8, w[f * kWave]),
                                                         __builtin_bit_cast(prod_bf16x8, xs), acc[f], 0, 0, 0);
    }
  };
  // The rows from .. to - 1.  A lane has, of row l16, columns 32 h + 8 group .. + 7 in the fragments 2 h and 2 h + 1.
  auto store = [&](const At& at, int64_t from, int64_t to) {
    const int64_t r = row0(at) + l16;
#pragma unroll
    for (int h = 0; h < kFragsN / 2; ++h) {
      const int c = n0 + h * 32 + group * 8;
      if (r < from || r >= to || c >= p.n) continue;
      uint16_t* out = p.y + r * p.n + c;
      float v[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = acc[2 * h][q];
        v[4 + q] = acc[2 * h + 1][q];
      }
      if (p.accumulate) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] += c + q < p.n ? to_float<uint16_t>(out[q]) : 0.f;
      }
      if (p.relu) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = relu(v[q]);
      }
      if (p.wide == 8) {
        store_vec<uint16_t, 8>(out, 0, v);
      } else if (p.wide == 4) {
        store_vec<uint16_t, 4>(out, 0, {v[0], v[1], v[2], v[3]});
        if (c + 4 < p.n) store_vec<uint16_t, 4>(out, 4, {v[4], v[5], v[6], v[7]});
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (c + q < p.n) out[q] = from_float<uint16_t>(v[q]);
      }
    }
  };
  At at{first, 0, 0};
  if (at.block >= p.row_blocks) return;
  load(at, x[0]);
  begin();
  auto turn = [&](ProdRaw<ODD> (&now)[kProdChunk], ProdRaw<ODD> (&ahead)[kProdChunk]) {   // false: that was the last one
    const At then = next(at);
    load(then, ahead);
    __builtin_amdgcn_sched_barrier(0);   // (those of this chunk are waited for alone)
    multiply(at, now);
    // Rows of the fragment without the second operand are stored before it comes: their zeros must not meet a weight that is
    // not finite.
    const bool ends = then.block != at.block, parts = then.which > at.which && row0(at) + 16 > p.a[1].rows;   // wave-uniform
    if (ends || parts) store(at, parts ? p.a[1].rows : 0, at.which == 1 ? p.a[1].rows : p.m);
    if (ends) {
      if (then.block >= p.row_blocks) return false;
      begin();
    }
    at = then;
    return true;
  };
  while (turn(x[0], x[1]) && turn(x[1], x[0])) {
  }
}

static int prod_steps(int64_t k) { return static_cast<int>(ceil_div(k, kProdStep)); }
static size_t prod_lds(int64_t steps, int wn) { return steps * kProdStep * 64 * wn * 2 + 64 * wn * sizeof(float); }
// Groups of 64 columns: the widest tile whose weights fit LDS; 0: none does.
static int prod_columns(int64_t n, int64_t steps) {
  for (int wn = n <= 64 ? 1 : n <= 128 ? 2 : 4; wn > 0; wn >>= 1)
    if (steps * kProdStep * 64 * wn * 2 <= kProdLds) return wn;
  return 0;
}

template <int WN>
static void launch_product(ProdParams& p, bool odd, hipStream_t st) {
  const size_t lds = prod_lds(p.a[0].steps + p.a[1].steps, WN);
  // as many turns of the loop over the rows for every workgroup of a launch that the CUs hold at once
  const int64_t most = std::max<int64_t>(kProdGroups / (lds > 80 * 1024 ? 2 : 1) / p.tiles_n, 1);
  p.walkers = static_cast<int>(ceil_div(p.row_blocks, ceil_div(p.row_blocks, most)));
  const dim3 grid(static_cast<unsigned>(ceil_div(static_cast<int64_t>(p.walkers) * p.tiles_n, 8) * 8)), block(kProdBlock);
  if (odd) hipLaunchKernelGGL((rows_product_kernel<WN, true>), grid, block, lds, st, p);
  else hipLaunchKernelGGL((rows_product_kernel<WN, false>), grid, block, lds, st, p);
}

}  // namespace apt

extern "C" int apt_rows_product_fits(int64_t m, int64_t n, int64_t k1, int64_t k2) {
  using namespace apt;
  return m >= 0 && m <= (int64_t{1} << 34) && n > 0 && n <= (1 << 16) && k1 > 0 && k2 >= 0 && k1 <= 4096 && k2 <= 4096 &&
         prod_columns(n, prod_steps(k1) + prod_steps(k2)) > 0;
}

extern "C" int apt_rows_product(const void* x1, int64_t k1, const void* w1, int64_t w1_stride_n, int64_t w1_stride_k,
                                const void* x2, int64_t k2, const void* w2, int64_t w2_stride_n, int64_t w2_stride_k,
                                int64_t m, int64_t m2, int64_t n, const void* bias, int accumulate, int relu, void* y,
                                void* stream) {
  using namespace apt;
  APT_REQUIRE(apt_rows_product_fits(m, n, k1, k2) && m2 >= 0 && m2 <= m, APT_ELIMIT,
              "apt_rows_product: sizes out of range (m %lld, m2 %lld, n %lld, k %lld + %lld)", (long long)m, (long long)m2,
              (long long)n, (long long)k1, (long long)k2);
  if (m == 0) return APT_OK;
  APT_REQUIRE(x1 != nullptr && w1 != nullptr && y != nullptr && (k2 == 0 || (w2 != nullptr && (m2 == 0 || x2 != nullptr))),
              APT_EINVAL, "apt_rows_product: a tensor is NULL");
  // (a stride of a side of one element is not looked at)
  const auto plain = [&](int64_t k, int64_t sn, int64_t sk) {
    return (k == 1 || sk == 1) ? (n == 1 || (sn >= k && (n + 256) * sn <= (1 << 30)))
                               : ((n == 1 || sn == 1) && sk >= n && (k + 32) * sk <= (1 << 30));
  };
  APT_REQUIRE(plain(k1, w1_stride_n, w1_stride_k) && (k2 == 0 || plain(k2, w2_stride_n, w2_stride_k)), APT_EINVAL,
              "apt_rows_product: weights must be contiguous along one side");
  ProdParams p{};
  bool odd = false;
  const auto operand = [&](const void* x, int64_t k, const void* w, int64_t sn, int64_t sk, int64_t rows) {
    ProdOperand a{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), rows, static_cast<int>(k),
                  k > 0 ? prod_steps(k) : 0, sn, sk};
    if (k == 1) a.stride_k = 1;
    if (n == 1) a.stride_n = a.stride_k == 1 ? std::max<int64_t>(k, 1) : 1;
    const int64_t pitch = a.stride_k == 1 ? a.stride_n : a.stride_k;
    odd |= k > 0 && (k % 2 != 0 || (pitch % 2 != 0) ||
                     ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 3) != 0);
    return a;
  };
  p.a[0] = operand(x1, k1, w1, w1_stride_n, w1_stride_k, m);
  p.a[1] = operand(x2, k2, w2, w2_stride_n, w2_stride_k, m2);
  if (m2 == 0) p.a[1].steps = 0;
  p.m = m;
  p.n = static_cast<int>(n);
  p.bias = static_cast<const uint16_t*>(bias);
  p.accumulate = accumulate;
  p.relu = relu;
  p.y = static_cast<uint16_t*>(y);
  const uintptr_t at = reinterpret_cast<uintptr_t>(y);
  p.wide = n % 8 == 0 && (at & 15) == 0 ? 8 : n % 4 == 0 && (at & 7) == 0 ? 4 : 1;
  p.row_blocks = ceil_div(m, kProdRows);
  int wn = prod_columns(n, p.a[0].steps + p.a[1].steps);
  while (wn > 1 && p.row_blocks * ceil_div(n, 64 * wn) < 256) wn >>= 1;   // (a workgroup for every CU)
  p.tiles_n = static_cast<int>(ceil_div(n, 64 * wn));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (wn == 1) launch_product<1>(p, odd, st);
  else if (wn == 2) launch_product<2>(p, odd, st);
  else launch_product<4>(p, odd, st);
  APT_LAUNCH_CHECK("rows_product_kernel");
  return APT_OK;
}

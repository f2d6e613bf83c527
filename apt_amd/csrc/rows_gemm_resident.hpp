// fp32 products of a layer's rows (rows_gemm.hip) whose weights fit LDS, split: a workgroup splits those of its column tile
// there once and keeps them while its wavefronts walk over their share of the rows, 16 MF at a time and all columns of the
// tile.  The rows go from memory into registers, two steps of the product ahead, and are split there by the wavefront that
// multiplies them: no barrier after the weights, so that wavefronts read, split, multiply and write at different times.
#pragma once

#include "common.hpp"
#include "feature_rows.hpp"
#include "split_bf16.hpp"

namespace apt {

constexpr int kResWaves = 8;
constexpr int kResBlock = kResWaves * kWave;
constexpr int kResChunk = 2;               // steps whose rows are loaded together
constexpr int kResMF = 2;                  // row fragments of a wavefront
constexpr int kResRows = kResWaves * kResMF * 16;
using res_buffer_t = __amdgpu_buffer_rsrc_t;

struct ResidentParams {
  GemmParams g;
  int steps1, steps2, tiles_n, walkers;   // walkers: workgroups of a column tile
  int64_t row_blocks;
};

// NF: column fragments of the tile.
template <int NF>
__global__ __launch_bounds__(kResBlock, 2) void rows_gemm_resident_kernel(ResidentParams p) {
  constexpr int kPartVecs = NF * kWave;
  extern __shared__ __align__(16) gemm_u32x4 s_weights[];   // [step][part][column fragment][lane]
  const GemmParams& g = p.g;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l16 = lane % 16, group = lane / 16;
  // The workgroups of the same rows (other columns) follow each other on one XCD.
  const int i = static_cast<int>(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8);
  const int64_t first = __builtin_amdgcn_readfirstlane(i / p.tiles_n), stride = p.walkers;
  const int tile = __builtin_amdgcn_readfirstlane(i % p.tiles_n);
  if (first >= stride) return;   // block-uniform (the grid is a multiple of eight)
  const int64_t n0 = static_cast<int64_t>(tile) * NF * 16;
  const int steps = p.steps1 + p.steps2;
  constexpr int kBatch = 4;
  const int all = steps * kPartVecs;
  for (int j0 = threadIdx.x; j0 < all; j0 += kBatch * kResBlock) {   // a thread per lane of a fragment, kBatch on their way
    float v[kBatch][8];
    auto place = [&](int u, int& step, int& f, int& at, int64_t& n, int64_t& k0, int64_t& depth) {
      const int j = min(j0 + u * kResBlock, all - 1);
      step = j / kPartVecs;
      f = j % kPartVecs / kWave;
      at = j % kWave;
      const bool one = step < p.steps1;
      n = n0 + f * 16 + at % 16;
      k0 = static_cast<int64_t>(one ? step : step - p.steps1) * kGemmStep + at / 16 * 8;
      depth = one ? g.k1 : g.k2;
      return one;
    };
    int step, f, at;
    int64_t n, k0, depth;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const bool one = place(u, step, f, at, n, k0, depth);
      const float* w = one ? g.w1.w : g.w2.w;
      const int64_t sn = one ? g.w1.stride_n : g.w2.stride_n, sk = one ? g.w1.stride_k : g.w2.stride_k;
#pragma unroll
      for (int e = 0; e < 8; ++e)   // (the address of a missing element is one that exists)
        v[u][e] = w[min(n, g.n - 1) * sn + min(k0 + e, depth - 1) * sk];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      place(u, step, f, at, n, k0, depth);
      if (j0 + u * kResBlock >= all) continue;
      gemm_u32x4 part[kGemmParts];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const bool in0 = n < g.n && k0 + 2 * d < depth, in1 = n < g.n && k0 + 2 * d + 1 < depth;
        const SplitPair s = split_pair(in0 ? v[u][2 * d] : 0.f, in1 ? v[u][2 * d + 1] : 0.f);
        part[0][d] = s.hi;
        part[1][d] = s.mid;
        part[2][d] = s.lo;
      }
#pragma unroll
      for (int q = 0; q < kGemmParts; ++q) s_weights[(step * kGemmParts + q) * kPartVecs + f * kWave + at] = part[q];
    }
  }
  __syncthreads();
  // (no barriers below)
  // The wavefront's work is a sequence of chunks of kResChunk steps: of the first operand, then of the second, then of the
  // next tile of rows.
  struct At {
    int64_t block;
    int which, step;
  };
  auto row0 = [&](const At& at) { return at.block * kResRows + wave * (kResMF * 16); };
  auto steps_of = [&](const At& at) { return at.which == 0 ? p.steps1 : p.steps2; };
  auto depth_of = [&](const At& at) { return static_cast<int>(at.which == 0 ? g.k1 : g.k2); };
  auto next = [&](At at) {
    at.step += kResChunk;
    if (at.step >= steps_of(at)) {
      at.step = 0;
      if (at.which == 0 && p.steps2 > 0 && row0(at) < g.m2) {
        at.which = 1;
      } else {
        at.which = 0;
        at.block += stride;
      }
    }
    return at;
  };
  gemm_f32x4 x[2][kResMF][kResChunk][2];
  auto load = [&](const At& at, gemm_f32x4 (&v)[kResMF][kResChunk][2]) {
    const int64_t rows = at.which == 0 ? g.m : g.m2, row = min(row0(at), rows);   // (past the end: an empty range)
    const int depth = depth_of(at);
    const float* base = (at.which == 0 ? g.x1 : g.x2) + row * depth;
    const res_buffer_t buffer = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(base), 0, static_cast<uint32_t>(min(rows - row, static_cast<int64_t>(kResMF * 16)) * depth * 4), 0x00020000);
#pragma unroll
    for (int m = 0; m < kResMF; ++m)
#pragma unroll
      for (int s = 0; s < kResChunk; ++s) {
        const uint32_t to = static_cast<uint32_t>(((m * 16 + l16) * depth + (at.step + s) * kGemmStep + group * 8) * 4) |
                            (at.step + s < steps_of(at) ? 0u : 0x80000000u);   // (behind the last step: nothing is read)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[m][s][h] = __builtin_bit_cast(gemm_f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer, to + 16 * h, 0, 0));
      }
  };
  gemm_f32x4 acc[kResMF][NF];
  auto clear = [&]() {
#pragma unroll
    for (int m = 0; m < kResMF; ++m)
#pragma unroll
      for (int f = 0; f < NF; ++f) acc[m][f] = gemm_f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto multiply = [&](const At& at, gemm_f32x4 (&v)[kResMF][kResChunk][2]) {
    const int base = at.which == 0 ? 0 : p.steps1;
#pragma unroll
    for (int s = 0; s < kResChunk; ++s) {
      if (at.step + s >= steps_of(at)) continue;   // wave-uniform
      const int left = depth_of(at) - (at.step + s) * kGemmStep - group * 8;
      gemm_u32x4 xs[kResMF][kGemmParts];
#pragma unroll
      for (int m = 0; m < kResMF; ++m)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          float a = v[m][s][d / 2][d % 2 * 2], b = v[m][s][d / 2][d % 2 * 2 + 1];
          if (at.step + s + 1 == steps_of(at)) {   // (reaches into the next row)
            a = 2 * d < left ? a : 0.f;
            b = 2 * d + 1 < left ? b : 0.f;
          }
          const SplitPair t = split_pair(a, b);
          xs[m][0][d] = t.hi;
          xs[m][1][d] = t.mid;
          xs[m][2][d] = t.lo;
        }
      const gemm_u32x4* w = s_weights + (base + at.step + s) * kGemmParts * kPartVecs + lane;
#pragma unroll
      for (int f0 = 0; f0 < NF; f0 += 2) {
        gemm_u32x4 ws[2][kGemmParts];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int q = 0; q < kGemmParts; ++q) ws[f][q] = w[q * kPartVecs + (f0 + f) * kWave];
        // A step's products are added up on their own, the small ones first: one rounding of the long sum per step
        gemm_f32x4 sum[2][kResMF];
#pragma unroll
        for (int t = 0; t < kSplitProducts; ++t)
#pragma unroll
          for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int m = 0; m < kResMF; ++m)
              sum[f][m] = gemm_mfma(ws[f][kSplitA[t]], xs[m][kSplitB[t]], t == 0 ? gemm_f32x4{0.f, 0.f, 0.f, 0.f} : sum[f][m]);
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int m = 0; m < kResMF; ++m) acc[m][f0 + f] += sum[f][m];
      }
    }
  };
  // A lane has four consecutive columns of row l16 of its fragment.
  auto store = [&](const At& at) {
    bool finite = true;
#pragma unroll
    for (int m = 0; m < kResMF; ++m)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int q = 0; q < 4; ++q) finite &= __builtin_isfinite(acc[m][f][q]);
    if (__any(!finite)) gemm_again<kResMF, NF>(g, row0(at), n0, acc);
#pragma unroll
    for (int m = 0; m < kResMF; ++m) gemm_store<NF>(g, row0(at) + m * 16 + l16, n0, acc[m]);
  };
  At at{first, 0, 0};
  if (at.block >= p.row_blocks) return;
  load(at, x[0]);
  clear();
  auto turn = [&](gemm_f32x4 (&now)[kResMF][kResChunk][2], gemm_f32x4 (&ahead)[kResMF][kResChunk][2]) {   // false: that was the last one
    const At then = next(at);
    load(then, ahead);
    __builtin_amdgcn_sched_barrier(0);   // (those of this chunk are waited for alone)
    multiply(at, now);
    if (then.block != at.block) {
      store(at);
      if (then.block >= p.row_blocks) return false;
      clear();
    }
    at = then;
    return true;
  };
  while (turn(x[0], x[1]) && turn(x[1], x[0])) {
  }
}

static int64_t resident_bytes(int64_t steps, int nf) { return steps * nf * kGemmParts * kWave * 16; }   // (96 KB at the most)
// Turns of the loop over the rows: as many for every workgroup of a launch that the 256 CUs hold at once.
static int64_t resident_turns(int64_t row_blocks, int64_t tiles_n) {
  return ceil_div(row_blocks, std::max<int64_t>(256 / tiles_n, 1));
}
// Column fragments of a tile; 0: the kernel without resident weights is the better one.  That is so
//   for more than four steps, whose weights leave room for 64 columns only, so that the rows are read and split once for each
//     (26 k rows, 256 -> 256: 32 us there, 40 here);
//   where the launch leaves many CUs idle, or has one turn only to pay for its weights with (the share of the CUs' turns that
//     has work / turns; us here / there: 128 -> 256 26 k rows 0.8 / 1 26 / 21, 49 k 0.75 / 2 35 / 31, 53 k 0.81 / 2 35 / 35, 124 k
//     0.95 / 4 57 / 63, 460 k 202 / 238; 100 -> 512 16 k 0.98 / 1 22 / 22, 26 k 0.8 / 2 32 / 35; 128 -> 1000 40 k 70 / 77);
//   not so much for narrow results of few steps or of rows that begin inside a line, which the other kernel reads in more
//     pieces (50 -> 100 32 k rows 0.5 / 1 14 / 13, 40 k 0.61 / 1 14 / 17, 124 k 22 / 33; 64 -> 64 100 k 0.76 / 2 17 / 22; 128 -> 128 as
//     the wide ones, 65 k 1 / 1 27 / 26, 124 k 37 / 43);
//   for a last tile that is nearly empty (128 -> 385, 100 k rows 148 / 129; 128 -> 300 65 / 81, 128 -> 301 106 / 121).
// Up to 32 columns it is the better one throughout (100 -> 16: 5 k rows 10 / 13, 200 k 25 / 42).
static int resident_columns(int64_t m, int64_t n, int64_t steps, bool broken) {   // broken: rows begin inside a line
  if (steps > 4) return 0;
  if (n <= 32) return 2;
  const int nf = n <= 64 ? 4 : 8;
  const int64_t tiles = ceil_div(n, nf * 16), row_blocks = ceil_div(m, kResRows), turns = resident_turns(row_blocks, tiles);
  const double busy = static_cast<double>(row_blocks * tiles) / static_cast<double>(256 * turns);
  if (n <= 128 && (steps <= 2 || broken)) return busy >= 0.6 ? nf : 0;
  return turns >= 2 && busy >= 0.78 && n * 100 >= tiles * nf * 16 * 77 ? nf : 0;
}

template <int NF>
static void launch_resident(ResidentParams& p, hipStream_t st) {
  p.tiles_n = static_cast<int>(ceil_div(p.g.n, NF * 16));
  p.row_blocks = ceil_div(p.g.m, kResRows);
  const size_t lds = resident_bytes(p.steps1 + p.steps2, NF);
  p.walkers = static_cast<int>(ceil_div(p.row_blocks, resident_turns(p.row_blocks, p.tiles_n)));
  const int64_t grid = ceil_div(static_cast<int64_t>(p.walkers) * p.tiles_n, 8) * 8;
  hipLaunchKernelGGL((rows_gemm_resident_kernel<NF>), dim3(static_cast<unsigned>(grid)), dim3(kResBlock), lds, st, p);
}

}  // namespace apt

// The dense product of a layer over a block's rows in fp32, two operand pairs at once:
//   y[r, :] = x1[r, :] w1^T + x2[r, :] w2^T + bias        (x2 for the first m2 rows only)
//
// A GraphSAGE layer is the sum of two such products and its gradient towards the features is another; one pass
// over the result saves writing one product, adding the other and, backward, a zero-filled copy of the rows.
//
// fp32 operands are split into three bf16 parts (split_bf16.hpp) and multiplied on the bf16 matrix units with fp32
// accumulators: six products take less than half the time of the fp32 matrix instruction, whose rate (157 TFLOP/s, one
// sixteenth of bf16's) bounds these products otherwise.  A result that is not finite is formed again with that
// instruction.
//
// Tile: a workgroup has 64 x (64 or 16) result elements per wavefront; the rows go through LDS, already split (every
// wavefront of a row range shares them), and the weights come from the workspace, where rows_gemm_weights_kernel left
// them split and in the order of the MFMA operand: a few hundred KB that all workgroups read from the L2.
//
// Measured (both launches; the library's products and the addition where there are two), error against 64 bits:
//   170 k rows, 100 + 100 -> 256    173 us / 449 us    6e-8 / 1.5e-7
//   40 k rows, 256 -> 256            50 /  57          6e-8 / 2.0e-7
//   170 k rows, 256 -> 47            76 /  75          5e-8 / 1.9e-7
//   1 k rows, 256 + 256 -> 47        22 /  42          8e-8 / 2.4e-7
// The first has 46 us on the matrix units at their rate and 310 MB of rows and results (55 us); in the layers' passes the
// matrix units work 39 % of this kernel's cycles and the vector units, which split, 33 %: the workgroups of a launch read,
// multiply and write much in step.  Where the weights fit LDS: rows_gemm_resident.hpp (460 k rows, 100 -> 256 212 us, 230 here).
#include <algorithm>

#include "common.hpp"
#include "feature_rows.hpp"
#include "split_bf16.hpp"

namespace apt {

typedef float gemm_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t gemm_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t gemm_u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kGemmStep = 32;      // depth of a bf16 MFMA
constexpr int kGemmWaves = 4;
constexpr int kGemmBlock = kGemmWaves * kWave;
constexpr int kGemmFragsN = 4;     // 64 columns per wavefront
constexpr int kGemmAhead = 2;      // steps whose rows are on their way
constexpr int kGemmParts = 3;

struct GemmWeight {
  const float* w;
  int64_t stride_n, stride_k;
};

struct GemmParams {
  const float* x1;
  const float* x2;
  int64_t k1, k2, m, m2, n;
  GemmWeight w1, w2;
  const gemm_u32x4* parts;   // [step][column fragment][part][lane]
  int frags;                 // column fragments: ceil(n / 64) * 4
  const float* bias;
  int accumulate, relu;
  float* y;
};

__device__ __forceinline__ float gemm_weight(const GemmParams& p, int64_t n, int64_t k) {
  if (n >= p.n) return 0.f;
  if (k < p.k1) return p.w1.w[n * p.w1.stride_n + k * p.w1.stride_k];
  k -= p.k1;
  return k < p.k2 ? p.w2.w[n * p.w2.stride_n + k * p.w2.stride_k] : 0.f;
}

// A thread per lane of a fragment: eight consecutive k of one column.
__global__ __launch_bounds__(kGemmBlock) void rows_gemm_weights_kernel(GemmParams p, int steps, gemm_u32x4* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kGemmBlock + threadIdx.x;
  if (i >= static_cast<int64_t>(steps) * p.frags * kWave) return;
  const int lane = static_cast<int>(i % kWave);
  const int64_t frag = i / kWave;
  const int64_t n = frag % p.frags * 16 + lane % 16;
  const int64_t k = frag / p.frags * kGemmStep + lane / 16 * 8;
  gemm_u32x4 part[kGemmParts];
  float w[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {   // all on their way together: the address of a missing element is one that exists
    const bool first = k + j < p.k1, in = n < p.n && k + j < p.k1 + p.k2;
    const int64_t kj = first ? k + j : k + j - p.k1;
    const float* at = first ? p.w1.w + n * p.w1.stride_n + kj * p.w1.stride_k : p.w2.w + n * p.w2.stride_n + kj * p.w2.stride_k;
    w[j] = *(in ? at : p.w1.w);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bool in0 = n < p.n && k + 2 * j < p.k1 + p.k2, in1 = n < p.n && k + 2 * j + 1 < p.k1 + p.k2;
    const SplitPair s = split_pair(in0 ? w[2 * j] : 0.f, in1 ? w[2 * j + 1] : 0.f);
    part[0][j] = s.hi;
    part[1][j] = s.mid;
    part[2][j] = s.lo;
  }
#pragma unroll
  for (int q = 0; q < kGemmParts; ++q) out[(frag * kGemmParts + q) * kWave + lane] = part[q];
}

__device__ __forceinline__ gemm_f32x4 gemm_mfma(gemm_u32x4 a, gemm_u32x4 b, gemm_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gemm_bf16x8, a), __builtin_bit_cast(gemm_bf16x8, b), c, 0,
                                                 0, 0);
}

// Fragments of rows row0 .. and columns n0 .. with the fp32 instruction.
template <int MF, int NF>
__device__ __forceinline__ void gemm_again(const GemmParams& p, int64_t row0, int64_t n0, gemm_f32x4 (&acc)[MF][NF]) {
  const int l16 = threadIdx.x % 16, group = threadIdx.x % kWave / 16;
#pragma unroll 1
  for (int t = 0; t < MF * NF; ++t) {
    const int m = t / NF, f = t % NF;
    const int64_t r = row0 + m * 16 + l16, n = n0 + f * 16 + l16;
    // the operands apart: zeros in the place of a missing second row must not meet an infinite weight
    gemm_f32x4 c = {0.f, 0.f, 0.f, 0.f}, c2 = {0.f, 0.f, 0.f, 0.f};
    for (int64_t k0 = 0; k0 < p.k1; k0 += 4) {
      const int64_t k = k0 + group;
      const bool in = k < p.k1;
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? gemm_weight(p, n, k) : 0.f, in && r < p.m ? p.x1[r * p.k1 + k] : 0.f, c, 0, 0, 0);
    }
    for (int64_t k0 = 0; k0 < (row0 < p.m2 ? p.k2 : 0); k0 += 4) {
      const int64_t k = k0 + group;
      const bool in = k < p.k2;
      c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? gemm_weight(p, n, p.k1 + k) : 0.f,
                                                in && r < p.m2 ? p.x2[r * p.k2 + k] : 0.f, c2, 0, 0, 0);
    }
    if (r < p.m2) c += c2;
#pragma unroll
    for (int mm = 0; mm < MF; ++mm)
#pragma unroll
      for (int ff = 0; ff < NF; ++ff)
        if (mm == m && ff == f) acc[mm][ff] = c;
  }
}
// Row r of fragments of columns n0 ..: a lane has four consecutive columns of each.
template <int NF>
__device__ __forceinline__ void gemm_store(const GemmParams& p, int64_t r, int64_t n0, const gemm_f32x4 (&acc)[NF]) {
  const int group = threadIdx.x % kWave / 16;
  const bool wide = p.n % 4 == 0;
  if (r >= p.m) return;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int64_t n = n0 + f * 16 + group * 4;
    float* out = p.y + r * p.n + n;
    if (wide) {
      if (n >= p.n) continue;
      gemm_f32x4 v = acc[f];
      if (p.bias != nullptr) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] += p.bias[n + q];
      }
      if (p.accumulate) v += *reinterpret_cast<const gemm_f32x4*>(out);
      if (p.relu) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = relu(v[q]);
      }
      *reinterpret_cast<gemm_f32x4*>(out) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (n + q >= p.n) continue;
        float v = acc[f][q];
        if (p.bias != nullptr) v += p.bias[n + q];
        if (p.accumulate) v += out[q];
        if (p.relu) v = relu(v);
        out[q] = v;
      }
    }
  }
}

// WN wavefronts side by side along the columns, the others along the rows; MF row fragments (of 16) per wavefront.
// VEC: rows are read four elements at a time (k1, k2 multiples of four, aligned) or one.
template <int WN, int MF, int VEC>
__global__ __launch_bounds__(kGemmBlock, 2) void rows_gemm_kernel(GemmParams p) {
  constexpr int kFragsM = kGemmWaves / WN * MF;                            // row fragments of the workgroup
  constexpr int kRows = kFragsM * 16;
  constexpr int kChunks = kRows * (kGemmStep / 4);                         // four elements each
  constexpr int kPerThread = (kChunks + kGemmBlock - 1) / kGemmBlock;
  __shared__ __align__(16) uint32_t s_x[2][kGemmParts][kFragsM * kWave * 4];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int l16 = lane % 16, group = lane / 16;
  const int wn = wave % WN, wm = wave / WN;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRows;
  const int frag_n = (blockIdx.y * WN + wn) * kGemmFragsN;                 // first column fragment of the wavefront
  const bool active = frag_n < p.frags;                                    // wave-uniform
  const int64_t depth = p.k1 + (row0 < p.m2 ? p.k2 : 0);
  const int steps = static_cast<int>((depth + kGemmStep - 1) / kGemmStep);

  // What a thread reads of a step; an element outside the operands is read from the start of x1 and replaced by zero
  // when it is used (a branch around a load would wait for it).
  auto source = [&](int step, int i, int j, bool& in) -> const float* {
    const int c = tid + i * kGemmBlock;
    const int64_t r = row0 + c / 8;
    const int64_t k = static_cast<int64_t>(step) * kGemmStep + c % 8 * 4 + j;
    const bool first = k < p.k1;
    in = (kChunks % kGemmBlock == 0 || c < kChunks) && k < depth && r < (first ? p.m : p.m2);
    const float* at = first ? p.x1 + r * p.k1 + k : p.x2 + r * p.k2 + (k - p.k1);
    return in ? at : p.x1;
  };
  float ahead[kGemmAhead][kPerThread][4];
  auto load = [&](int step, float (&v)[kPerThread][4]) {
    bool in;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      if constexpr (VEC == 4) {
        const gemm_f32x4 t = *reinterpret_cast<const gemm_f32x4*>(source(step, i, 0, in));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = t[j];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = *source(step, i, j, in);
      }
    }
  };
  auto stage = [&](int step, const float (&v)[kPerThread][4]) {
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const int c = tid + i * kGemmBlock;
      float t[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bool in;
        source(step, i, VEC == 4 ? 0 : j, in);
        t[j] = in ? v[i][j] : 0.f;
      }
      if (kChunks % kGemmBlock != 0 && c >= kChunks) continue;
      const int row = c / 8, q = c % 8;
      const int at = ((row / 16 * 4 + q / 2) * 16 + row % 16) * 4 + (q & 1) * 2;
      const SplitPair a = split_pair(t[0], t[1]), b = split_pair(t[2], t[3]);
      uint32_t(*buf)[kFragsM * kWave * 4] = s_x[step & 1];
      *reinterpret_cast<gemm_u32x2*>(&buf[0][at]) = gemm_u32x2{a.hi, b.hi};
      *reinterpret_cast<gemm_u32x2*>(&buf[1][at]) = gemm_u32x2{a.mid, b.mid};
      *reinterpret_cast<gemm_u32x2*>(&buf[2][at]) = gemm_u32x2{a.lo, b.lo};
    }
  };
  gemm_u32x4 w[2][kGemmFragsN][kGemmParts];
  auto load_weights = [&](int step, gemm_u32x4 (&v)[kGemmFragsN][kGemmParts]) {
    const int frag = active ? frag_n : 0;                                  // (an idle wavefront's are not used)
    const gemm_u32x4* src =
        p.parts + (static_cast<int64_t>(min(step, steps - 1)) * p.frags + frag) * kGemmParts * kWave + lane;
#pragma unroll
    for (int f = 0; f < kGemmFragsN; ++f)
#pragma unroll
      for (int q = 0; q < kGemmParts; ++q) v[f][q] = src[(f * kGemmParts + q) * kWave];
  };
  gemm_f32x4 acc[MF][kGemmFragsN] = {};
  auto multiply = [&](int buf, const gemm_u32x4 (&v)[kGemmFragsN][kGemmParts]) {
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      gemm_u32x4 x[kGemmParts];
#pragma unroll
      for (int q = 0; q < kGemmParts; ++q)
        x[q] = *reinterpret_cast<const gemm_u32x4*>(&s_x[buf][q][((wm * MF + m) * kWave + lane) * 4]);
      // A step's products are added up on their own, the small ones first: one rounding of the long sum per step
      gemm_f32x4 sum[kGemmFragsN];
#pragma unroll
      for (int t = 0; t < kSplitProducts; ++t)
#pragma unroll
        for (int f = 0; f < kGemmFragsN; ++f)
          sum[f] = gemm_mfma(v[f][kSplitA[t]], x[kSplitB[t]], t == 0 ? gemm_f32x4{0.f, 0.f, 0.f, 0.f} : sum[f]);
#pragma unroll
      for (int f = 0; f < kGemmFragsN; ++f) acc[m][f] += sum[f];
    }
  };

  // Step s: its rows are in LDS buffer s % 2, its weights in registers; the rows of the next step are split into the
  // other buffer, those of later ones are on their way.
  if (steps > 0) {
#pragma unroll
    for (int a = 0; a < kGemmAhead; ++a) load(a, ahead[a]);
    load_weights(0, w[0]);
    stage(0, ahead[0]);
    load(kGemmAhead, ahead[0]);
    __syncthreads();
    for (int s0 = 0; s0 < steps; s0 += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int s = s0 + u;
        load_weights(s + 1, w[(u + 1) & 1]);
        if (active && s < steps) multiply(u, w[u]);                        // wave-uniform; loads stay outside
        stage(s + 1, ahead[(u + 1) & 1]);
        load(s + 1 + kGemmAhead, ahead[(u + 1) & 1]);
        __syncthreads();
      }
    }
  }
  if (!active) return;                                                     // no barriers below

  bool finite = true;
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < kGemmFragsN; ++f)
#pragma unroll
      for (int q = 0; q < 4; ++q) finite &= __builtin_isfinite(acc[m][f][q]);
  if (__any(!finite)) gemm_again<MF, kGemmFragsN>(p, row0 + wm * MF * 16, static_cast<int64_t>(frag_n) * 16, acc);
#pragma unroll
  for (int m = 0; m < MF; ++m) gemm_store<kGemmFragsN>(p, row0 + (wm * MF + m) * 16 + l16, static_cast<int64_t>(frag_n) * 16, acc[m]);
}

}  // namespace apt

#include "rows_gemm_resident.hpp"

namespace apt {

// The sum of two products that the library formed, with the ReLU: one pass instead of two.
template <typename T, int VEC>
__global__ __launch_bounds__(kGemmBlock) void add_rows_kernel(T* __restrict__ y, const T* __restrict__ x, int64_t vecs,
                                                              int act) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kGemmBlock + threadIdx.x; i < vecs;
       i += static_cast<int64_t>(gridDim.x) * kGemmBlock) {
    float a[VEC], b[VEC];
    load_vec<T, VEC>(y, i * VEC, a);
    load_vec<T, VEC>(x, i * VEC, b);
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      a[k] += b[k];
      if (act) a[k] = relu(a[k]);
    }
    store_vec<T, VEC>(y, i * VEC, a);
  }
}

template <typename T, int VEC>
static void launch_add_rows(void* y, const void* x, int64_t count, int act, hipStream_t st) {
  const int64_t vecs = count / VEC;
  hipLaunchKernelGGL((add_rows_kernel<T, VEC>), dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(vecs, kGemmBlock), 1 << 16))),
                     dim3(kGemmBlock), 0, st, static_cast<T*>(y), static_cast<const T*>(x), vecs, act);
}

static bool gemm_sizes_ok(int64_t m, int64_t m2, int64_t n, int64_t k1, int64_t k2) {
  return m >= 0 && m2 >= 0 && m2 <= m && n > 0 && n <= (1 << 16) && k1 > 0 && k1 <= (1 << 20) && k2 >= 0 && k2 <= (1 << 20) &&
         (n + 63) * (k1 + k2 + kGemmStep) <= (int64_t{1} << 28) && m <= (int64_t{1} << 34);
}
static int gemm_frags(int64_t n) { return static_cast<int>(ceil_div(n, 64) * kGemmFragsN); }

// 64 rows per wavefront (32 where fewer wavefronts share them: registers) if that leaves a workgroup for every CU; 16
// otherwise.
template <int WN, int VEC>
static void launch_gemm(const GemmParams& p, hipStream_t st) {
  const unsigned tiles_n = static_cast<unsigned>(ceil_div(p.frags / kGemmFragsN, WN));
  constexpr int64_t kRows = kGemmWaves / WN * 16;
  constexpr int kMost = WN == 4 ? 4 : 2;
  if (ceil_div(p.m, kMost * kRows) * tiles_n >= 256)
    hipLaunchKernelGGL((rows_gemm_kernel<WN, kMost, VEC>), dim3(static_cast<unsigned>(ceil_div(p.m, kMost * kRows)), tiles_n),
                       dim3(kGemmBlock), 0, st, p);
  else
    hipLaunchKernelGGL((rows_gemm_kernel<WN, 1, VEC>), dim3(static_cast<unsigned>(ceil_div(p.m, kRows)), tiles_n),
                       dim3(kGemmBlock), 0, st, p);
}

}  // namespace apt

extern "C" size_t apt_rows_gemm_workspace_bytes(int64_t n, int64_t k1, int64_t k2) {
  using namespace apt;
  if (!gemm_sizes_ok(0, 0, n, k1, k2)) return 0;
  return static_cast<size_t>(ceil_div(k1 + k2, kGemmStep)) * gemm_frags(n) * kGemmParts * kWave * sizeof(gemm_u32x4);
}

extern "C" int apt_rows_gemm(const float* x1, int64_t k1, const float* w1, int64_t w1_stride_n, int64_t w1_stride_k,
                             const float* x2, int64_t k2, const float* w2, int64_t w2_stride_n, int64_t w2_stride_k,
                             int64_t m, int64_t m2, int64_t n, const float* bias, int accumulate, int relu, float* y,
                             void* workspace, size_t workspace_bytes, void* stream) {
  using namespace apt;
  APT_REQUIRE(gemm_sizes_ok(m, m2, n, k1, k2), APT_ELIMIT, "apt_rows_gemm: sizes out of range (m %lld, m2 %lld, n %lld, k %lld + %lld)",
              (long long)m, (long long)m2, (long long)n, (long long)k1, (long long)k2);
  if (m == 0) return APT_OK;
  APT_REQUIRE(x1 != nullptr && w1 != nullptr && y != nullptr && (k2 == 0 || (w2 != nullptr && (m2 == 0 || x2 != nullptr))),
              APT_EINVAL, "apt_rows_gemm: a tensor is NULL");
  APT_REQUIRE(workspace != nullptr && workspace_bytes >= apt_rows_gemm_workspace_bytes(n, k1, k2) &&
                  (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
              APT_EWORKSPACE, "apt_rows_gemm: workspace too small or not 16-byte aligned (see apt_rows_gemm_workspace_bytes)");
  APT_REQUIRE(n % 4 != 0 || (reinterpret_cast<uintptr_t>(y) & 15) == 0, APT_EINVAL, "apt_rows_gemm: y is not 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  GemmParams p{x1, x2, k1, k2, m, k2 > 0 ? m2 : 0, n, {w1, w1_stride_n, w1_stride_k}, {w2, w2_stride_n, w2_stride_k},
               static_cast<const gemm_u32x4*>(workspace), gemm_frags(n), bias, accumulate, relu, y};
  const int64_t steps1 = ceil_div(k1, kGemmStep), steps2 = m2 > 0 ? ceil_div(k2, kGemmStep) : 0;
  if (const int nf = resident_columns(m, n, steps1 + steps2, k1 % 32 != 0 || (m2 > 0 && k2 % 32 != 0))) {
    ResidentParams q{p, static_cast<int>(steps1), static_cast<int>(steps2), 0, 0, 0};
    if (nf == 8) launch_resident<8>(q, st);
    else if (nf == 4) launch_resident<4>(q, st);
    else launch_resident<2>(q, st);
    APT_LAUNCH_CHECK("rows_gemm_resident_kernel");
    return APT_OK;
  }
  const int steps = static_cast<int>(ceil_div(k1 + k2, kGemmStep));
  hipLaunchKernelGGL(rows_gemm_weights_kernel,
                     dim3(static_cast<unsigned>(ceil_div(static_cast<int64_t>(steps) * p.frags * kWave, kGemmBlock))),
                     dim3(kGemmBlock), 0, st, p, steps, static_cast<gemm_u32x4*>(workspace));
  APT_LAUNCH_CHECK("rows_gemm_weights_kernel");
  const bool vec = k1 % 4 == 0 && k2 % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(x1) | reinterpret_cast<uintptr_t>(x2)) & 15) == 0;
  // wavefronts beside each other while there are columns for them
#define APT_ROWS_GEMM(WN)                   \
  if (vec) launch_gemm<WN, 4>(p, st);       \
  else launch_gemm<WN, 1>(p, st)
  if (n <= 64) { APT_ROWS_GEMM(1); }
  else if (n <= 128) { APT_ROWS_GEMM(2); }
  else { APT_ROWS_GEMM(4); }
#undef APT_ROWS_GEMM
  APT_LAUNCH_CHECK("rows_gemm_kernel");
  return APT_OK;
}

extern "C" int apt_add_rows(void* y, const void* x, int64_t count, int elem_size, int relu, void* stream) {
  using namespace apt;
  APT_REQUIRE(count >= 0 && (elem_size == 2 || elem_size == 4), APT_EINVAL, "apt_add_rows: count %lld, elem_size %d",
              (long long)count, elem_size);
  if (count == 0) return APT_OK;
  APT_REQUIRE(y != nullptr && x != nullptr, APT_EINVAL, "apt_add_rows: a tensor is NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool wide = ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
  if (elem_size == 4) {
    if (wide && count % 4 == 0) launch_add_rows<float, 4>(y, x, count, relu, st);
    else launch_add_rows<float, 1>(y, x, count, relu, st);
  } else {
    if (wide && count % 8 == 0) launch_add_rows<uint16_t, 8>(y, x, count, relu, st);
    else launch_add_rows<uint16_t, 1>(y, x, count, relu, st);
  }
  APT_LAUNCH_CHECK("add_rows_kernel");
  return APT_OK;
}

// Second half of a split reduction: sums of `splits` partial results in a fixed order.
#pragma once

#include "common.hpp"
#include "feature_rows.hpp"

namespace apt {

// out[e] = sum over s of part[s * stride + e], for up to three outputs that follow each other in a partial (any may
// be NULL: not wanted).  64 elements per workgroup, the splits dealt to its wavefronts.
constexpr int kPartialBlock = 1024;
constexpr int kPartialWaves = kPartialBlock / kWave;

struct PartialOutputs {
  void *a, *b, *c;
  int64_t na, nb, nc;
};

template <typename TA, typename TB>
__global__ __launch_bounds__(kPartialBlock) void partial_sums_kernel(const float* __restrict__ part, int64_t stride,
                                                                     int splits, PartialOutputs o) {
  constexpr int kUnroll = 8;
  __shared__ float s_sum[kPartialWaves][kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kWave + lane;
  const int64_t total = o.na + o.nb + o.nc;
  float sum = 0.f;
  if (e < total) {
    const float* src = part + e;
    for (int s = wave; s < splits; s += kPartialWaves * kUnroll) {
      float v[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int t = s + u * kPartialWaves;
        v[u] = t < splits ? src[static_cast<int64_t>(t) * stride] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) sum += v[u];
    }
  }
  s_sum[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || e >= total) return;
#pragma unroll
  for (int w = 1; w < kPartialWaves; ++w) sum += s_sum[w][lane];
  if (e < o.na) {
    if (o.a != nullptr) static_cast<TA*>(o.a)[e] = from_float<TA>(sum);
  } else if (e < o.na + o.nb) {
    if (o.b != nullptr) static_cast<TB*>(o.b)[e - o.na] = from_float<TB>(sum);
  } else if (o.c != nullptr) {
    static_cast<TB*>(o.c)[e - o.na - o.nb] = from_float<TB>(sum);
  }
}

template <typename TA, typename TB>
static void launch_partial_sums(const float* part, int64_t stride, int splits, void* a, int64_t na, void* b, int64_t nb,
                                void* c, int64_t nc, hipStream_t st) {
  const PartialOutputs o{a, b, c, na, nb, nc};
  hipLaunchKernelGGL((partial_sums_kernel<TA, TB>), dim3(static_cast<unsigned>(ceil_div(na + nb + nc, kWave))),
                     dim3(kPartialBlock), 0, st, part, stride, splits, o);
}

}  // namespace apt

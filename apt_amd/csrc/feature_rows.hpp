// Feature rows of the aggregation kernels: fp32 or bf16 (as bits) in memory, fp32 in registers.
#pragma once

#include "common.hpp"

namespace apt {

constexpr int kAggBlock = 256;
constexpr int kAggWaves = kAggBlock / kWave;

template <typename T> __device__ __forceinline__ float to_float(T v);
template <> __device__ __forceinline__ float to_float<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_float<uint16_t>(uint16_t v) {  // bf16 bits
  return __uint_as_float(static_cast<uint32_t>(v) << 16);
}

template <typename T> __device__ __forceinline__ T from_float(float v);
template <> __device__ __forceinline__ float from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ uint16_t from_float<uint16_t>(float v) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v));   // round to nearest even
}

// A value as it would be after being stored as a T and read back.
template <typename T> __device__ __forceinline__ float as_stored(float v) { return to_float<T>(from_float<T>(v)); }

template <typename T, int VEC> struct Pack;
template <> struct Pack<float, 4> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Pack<float, 1> { typedef float type; };
template <> struct Pack<float, 8> { typedef float type __attribute__((ext_vector_type(8))); };
template <> struct Pack<uint16_t, 4> { typedef uint16_t type __attribute__((ext_vector_type(4))); };
template <> struct Pack<uint16_t, 1> { typedef uint16_t type; };
template <> struct Pack<uint16_t, 8> { typedef uint16_t type __attribute__((ext_vector_type(8))); };

template <typename T, int VEC>
__device__ __forceinline__ void load_vec(const T* base, int64_t elem, float (&v)[VEC]) {
  using P = typename Pack<T, VEC>::type;
  const P raw = *reinterpret_cast<const P*>(base + elem);
  if constexpr (VEC == 1) {
    v[0] = to_float<T>(raw);
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = to_float<T>(raw[i]);
  }
}

// The same in two halves, for loads that should be in flight together: load every row from an address that is valid
// in any case (row 0 in the place of a missing one), then convert and use those that exist.  A load or a conversion
// inside a branch is waited for there.
template <typename T, int VEC> using Row = typename Pack<T, VEC>::type;
template <typename T, int VEC>
__device__ __forceinline__ Row<T, VEC> load_row(const T* base, int64_t elem) {
  return *reinterpret_cast<const Row<T, VEC>*>(base + elem);
}
template <typename T, int VEC>
__device__ __forceinline__ float row_elem(const Row<T, VEC>& raw, int k) {
  if constexpr (VEC == 1) return to_float<T>(raw);
  else return to_float<T>(raw[k]);
}

// max(v, 0) as torch has it: NaN stays NaN.
__device__ __forceinline__ float relu(float v) { return v < 0.f ? 0.f : v; }

template <typename T, int VEC>
__device__ __forceinline__ void store_vec(T* base, int64_t elem, const float (&v)[VEC]) {
  using P = typename Pack<T, VEC>::type;
  if constexpr (VEC == 1) {
    base[elem] = from_float<T>(v[0]);
  } else {
    P raw;
#pragma unroll
    for (int i = 0; i < VEC; ++i) raw[i] = from_float<T>(v[i]);
    *reinterpret_cast<P*>(base + elem) = raw;
  }
}

}  // namespace apt

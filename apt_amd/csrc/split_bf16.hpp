// fp32 values as sums of three bf16 (8 bits each, rounded to nearest): the products of the parts on the bf16 matrix units
// stand for an fp32 product.  Six of the nine are formed; those left out are below 2^-25 of the product.  (The low parts of
// a value below 2^-110 are subnormal bf16 or zero: such a value counts with fewer bits, down to the eight of its high part.)
// An infinity, or a value that rounds to one in bf16, has parts that are NaN: a result that is not finite is formed
// again in fp32.
#pragma once

#include "common.hpp"

namespace apt {

// Two fp32 values as three pairs of bf16.
struct SplitPair {
  uint32_t hi, mid, lo;
};
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  const bf16x2_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ SplitPair split_pair(float a, float b) {
  SplitPair s;
  s.hi = bf16_pair(a, b);
  a -= __uint_as_float(s.hi << 16);
  b -= __uint_as_float(s.hi & 0xffff0000u);
  s.mid = bf16_pair(a, b);
  a -= __uint_as_float(s.mid << 16);
  b -= __uint_as_float(s.mid & 0xffff0000u);
  s.lo = bf16_pair(a, b);
  return s;
}

// The six pairs of parts (0 = high), the small products first.
constexpr int kSplitProducts = 6;
constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0}, kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

}  // namespace apt

// fp32 values as sums of three bf16 (8 bits each, rounded to nearest): the products of the parts on the bf16 matrix units
// stand for an fp32 product.  Six of the nine are formed; those left out are below 2^-25 of the product.  (The low parts of
// a value below 2^-110 are subnormal bf16 or zero: such a value counts with fewer bits, down to the eight of its high part.)
// An infinity, or a value that rounds to one in bf16, has parts that are NaN: a result that is not finite is formed
// again in fp32.
#pragma once

#include "common.hpp"

namespace apt {

// Two fp32 values as three pairs of bf16.  Rounded by integer arithmetic (half away from zero): additions and masks issue
// at twice the rate of the conversion and of the shift that would take its result apart, 51 cycles a pair and wavefront
// instead of 71.  What is left after two parts has eight bits at the most and is cut off without loss.
struct SplitPair {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ uint32_t upper_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
__device__ __forceinline__ SplitPair split_pair(float a, float b) {
  SplitPair s;
  uint32_t x = __float_as_uint(a) + 0x8000u, y = __float_as_uint(b) + 0x8000u;
  s.hi = upper_halves(x, y);
  a -= __uint_as_float(x & 0xffff0000u);
  b -= __uint_as_float(y & 0xffff0000u);
  x = __float_as_uint(a) + 0x8000u;
  y = __float_as_uint(b) + 0x8000u;
  s.mid = upper_halves(x, y);
  a -= __uint_as_float(x & 0xffff0000u);
  b -= __uint_as_float(y & 0xffff0000u);
  s.lo = upper_halves(__float_as_uint(a), __float_as_uint(b));
  return s;
}

// The six pairs of parts (0 = high), the small products first.
constexpr int kSplitProducts = 6;
constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0}, kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

}  // namespace apt

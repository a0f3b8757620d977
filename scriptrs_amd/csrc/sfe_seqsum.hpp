// Sequential f32 sum of one value, as the reference's loops over a constant
// row add it up (src/frontend.rs:230-236), without walking the row.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace sfe {

__host__ __device__ __forceinline__ uint32_t seqsum_bits(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, sizeof u);
  return u;
}

// s = 0, then n times s = RN(s + a): the same bits as the loop, in about four
// additions per binade that the sum passes through (n = 2^30: about 100).
//
// Inside one binade the sum is a multiple m u of its ulp u, and an addition
// rounds m + |a| / u to an integer, ties to even.  Unless |a| / u ends in a
// half, that adds the same integer whatever m is.  If it does, the result is
// even, and from an even m the same even integer is added each time.  So from
// the second addition in a row that stays in one binade the mantissa grows by
// a constant, and all the steps up to the binade's end are one multiplication;
// the step across the end is a real addition again.  An addition that changes
// nothing never will (the sum is too large for a, or a is 0).
__host__ __device__ inline float sequential_sum(float a, int n) {
#pragma clang fp contract(off)
  float s = 0.0f;
  int inside = 0;  // additions in a row that stayed in the sum's binade
  for (int t = 0; t < n;) {
    const uint32_t p = seqsum_bits(s);
    s = s + a;
    ++t;
    const uint32_t b = seqsum_bits(s);
    if (b == p) return s;
    inside = (b >> 23) == (p >> 23) && (b & 0x7f800000u) != 0 ? inside + 1 : 0;
    if (inside < 2) continue;
    const uint32_t step = b - p;  // mantissas: the signs and exponents are equal
    const uint32_t left = (0x7fffffu - (b & 0x7fffffu)) / step;
    const uint32_t k = left < (uint32_t)(n - t) ? left : (uint32_t)(n - t);
    const uint32_t r = b + k * step;
    __builtin_memcpy(&s, &r, sizeof s);
    t += (int)k;
  }
  return s;
}

}  // namespace sfe

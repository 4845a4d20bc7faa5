// Division of element ordinals below 2^32 by a row width (Granlund and Montgomery, "Division by
// invariant integers using multiplication", 1994): with l = ceil(log2 C) and
// mul = floor(2^32 (2^l - C) / C) + 1, t = high half of mul n and n / C = (t + (n - t) / 2) >> (l - 1).
// Plain C++ so that the host tests can compare it with '/'.
#pragma once
#include <stdint.h>

namespace shk {

struct PwDivide {
  uint32_t mul, shift;
  int narrow;  // every ordinal fits 32 bits and C > 1
};
// For the ordinals of n elements in rows of C.
inline PwDivide pw_divide(int64_t n, int64_t C) {
  PwDivide d{0, 0, 0};
  if (C <= 1 || n > 0xffffffffll) return d;
  int l = 0;
  while ((1ll << l) < C) ++l;
  d.mul = (uint32_t)((((unsigned __int128)1 << 32) * (uint64_t)((1ll << l) - C)) / (uint64_t)C + 1);
  d.shift = (uint32_t)(l - 1);
  d.narrow = 1;
  return d;
}
__host__ __device__ inline uint32_t pw_quotient(uint32_t mul, uint32_t shift, uint32_t e) {
  const uint32_t h = (uint32_t)(((uint64_t)mul * e) >> 32);
  return (h + ((e - h) >> 1)) >> shift;
}

}  // namespace shk

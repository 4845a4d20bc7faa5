// Host build of synaptik_amd/csrc/pw_divide.h compared with '/': widths around powers of two, of 3
// to 5 and up to 2^32 - 1, at ordinals around multiples of the width and at the ends of the range.
// Prints "ok" or the first difference.
#define __host__
#define __device__
#include "../synaptik_amd/csrc/pw_divide.h"
#include <cstdio>
#include <vector>

int main() {
  std::vector<uint64_t> widths;
  for (int k = 1; k < 32; ++k)
    for (int d = -1; d <= 1; ++d) widths.push_back((1ull << k) + d);
  for (uint64_t c : {3ull, 5ull, 7ull, 641ull, 1001ull, 6700417ull, 2147483649ull, 4294967294ull, 4294967295ull})
    widths.push_back(c);
  uint64_t seed = 88172645463325252ull;
  for (int i = 0; i < 2000; ++i) {
    seed ^= seed << 13, seed ^= seed >> 7, seed ^= seed << 17;
    widths.push_back(2 + (seed >> (32 + i % 30)));
  }
  const uint64_t top = 0xffffffffull;
  for (uint64_t C : widths) {
    if (C < 2 || C > top) continue;
    const shk::PwDivide d = shk::pw_divide((int64_t)top, (int64_t)C);
    if (!d.narrow) return printf("FAIL %llu is not narrow\n", (unsigned long long)C), 1;
    for (int i = 0; i < 400; ++i) {
      seed ^= seed << 13, seed ^= seed >> 7, seed ^= seed << 17;
      const uint64_t q = i < 100 ? (uint64_t)i : i < 200 ? top / C - (i - 100) : seed % (top / C + 1);
      for (int o = -2; o <= 2; ++o) {
        const uint64_t e = q * C + (uint64_t)(int64_t)o;
        if (e > top) continue;  // (also where it would be negative)
        if (shk::pw_quotient(d.mul, d.shift, (uint32_t)e) != e / C)
          return printf("FAIL %llu / %llu\n", (unsigned long long)e, (unsigned long long)C), 1;
      }
    }
  }
  if (shk::pw_divide(1ll << 32, 7).narrow || shk::pw_divide(100, 1).narrow) return printf("FAIL range\n"), 1;
  printf("ok\n");
  return 0;
}

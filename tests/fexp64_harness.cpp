// Host build of synaptik_amd/csrc/fexp64.h checked against the library's binary64 functions
// rounded once to binary32, over every `stride`-th binary32 pattern.
// Prints for exp, tanh and sigmoid: evaluated differing max_ulp, then 1 if every NaN stays one
// and every zero keeps the library's sign.
#define __host__
#define __device__
#include "../synaptik_amd/csrc/fexp64.h"
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

static int64_t ordinal(float f) {
  int32_t i;
  memcpy(&i, &f, 4);
  return i < 0 ? -(int64_t)(i & 0x7fffffff) : (int64_t)i;
}
static double logistic(double x) {
  if (x >= 0.0) return 1.0 / (1.0 + exp(-x));
  const double e = exp(x);
  return e / (1.0 + e);
}

int main(int argc, char** argv) {
  const uint64_t stride = argc > 1 ? strtoull(argv[1], nullptr, 10) : 257;
  int ok = 1;
  for (int f = 0; f < 3; ++f) {
    int64_t n = 0, diff = 0, max_ulp = 0;
    for (uint64_t u = 0; u < 0x100000000ull; u += stride) {
      const uint32_t bits = (uint32_t)u;
      float t;
      memcpy(&t, &bits, 4);
      const double x = (double)t;
      const float got = f == 0 ? shk::exp_rn(t) : f == 1 ? shk::tanh_rn(t) : shk::sigmoid_rn(t);
      const float want = (float)(f == 0 ? exp(x) : f == 1 ? tanh(x) : logistic(x));
      if (std::isnan(want) || std::isnan(got)) {
        if (std::isnan(want) != std::isnan(got)) ok = 0;
        continue;
      }
      if (want == 0.0f && std::signbit(want) != std::signbit(got)) ok = 0;
      ++n;
      const int64_t d = llabs(ordinal(got) - ordinal(want));
      if (d) ++diff;
      if (d > max_ulp) max_ulp = d;
    }
    printf("%lld %lld %lld\n", (long long)n, (long long)diff, (long long)max_ulp);
  }
  printf("%d\n", ok);
  return 0;
}

// exp_fma_near against exp_fma for every stride-th float pattern of
// |x| <= kExpNear, and at the ends of the range: the number of differences.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "../../nest-gpu_amd/csrc/stepfactor.h"

static long differs(uint32_t u) {
  float x;
  memcpy(&x, &u, 4);
  if (!(std::fabs(x) <= ngpu::kExpNear)) return 0;
  const float a = ngpu::exp_fma(x), b = ngpu::exp_fma_near(x);
  return memcmp(&a, &b, 4) != 0;
}

int main() {
  long bad = 0;
  for (uint64_t u = 0; u < (1ull << 32); u += 509) bad += differs((uint32_t)u);
  for (float x : {0.0f, 88.5f, 88.73f, 100.0f, 100.1f, 103.9f, 104.0f, 110.0f, 110.1f, 150.0f, 1.0e6f})
    for (int d = -4; d <= 4; ++d) {
      uint32_t u;
      memcpy(&u, &x, 4);
      bad += differs(u + d) + differs((u + d) ^ 0x80000000u);
    }
  printf("%ld\n", bad);
  return bad != 0;
}

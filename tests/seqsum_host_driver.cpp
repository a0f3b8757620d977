// Host run of sequential_sum (scriptrs_amd/csrc/sfe_seqsum.hpp) against the
// loop it stands for, bit for bit: every n up to 20,000, then n up to 2^21 at
// random places, over values that end in a half ulp of a later binade (ties),
// short mantissas, both signs, the log-mel of digital silence, tiny values
// and 0; then long rows, which walked term by term would take hours.
//
// Prints "bad N" at the end (N values differed).
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <random>
#include <vector>

#include "sfe_seqsum.hpp"

static uint32_t bits(float f) {
  uint32_t u;
  memcpy(&u, &f, sizeof u);
  return u;
}

int main() {
  std::mt19937 rng(99);
  std::vector<float> v = {0.0f, -0.0f, 1.0f, 1.5f, 3.0f, -16.635532f, 16.635532f, 0.1f, 1e-12f, 1e-30f, 1e-39f, 3e-45f,
                          1e30f, 3e38f, INFINITY, -INFINITY};
  for (int i = 1; i <= 12; ++i) {  // 1 + odd multiples of small powers of two: ties a few binades on
    v.push_back(1.0f + ldexpf(1.0f, i - 24 + 1));
    v.push_back(-(1.0f + ldexpf(3.0f, i - 24 + 1)));
    v.push_back(1.0f + ldexpf((float)(2 * i + 1), -23));
  }
  std::uniform_real_distribution<float> ud(-20.0f, 64.0f);
  for (int i = 0; i < 40; ++i) v.push_back(ud(rng));
  for (int i = 0; i < 20; ++i) {  // squared deviations of constant rows
    const float d = ldexpf((float)(1 + rng() % 64), -20);
    v.push_back(d * d);
  }
  long bad = 0, checks = 0;
  for (float a : v) {
    float s = 0.0f;
    int next = 1;
    for (int n = 1; n <= 1 << 21; ++n) {
      s = s + a;
      if (n != next) continue;
      next = n < 20000 ? n + 1 : n + 1 + (int)(rng() % 8192);
      ++checks;
      if (bits(sfe::sequential_sum(a, n)) != bits(s)) {
        if (bad++ < 10) printf("a %a n %d: %a, loop %a\n", a, n, sfe::sequential_sum(a, n), s);
      }
    }
  }
  if (bits(sfe::sequential_sum(1.0f, 0)) != 0) ++bad;
  // rows of 2^30 terms: 1 stops growing at 2^24 (n + 1 rounds to even n)
  volatile float sink = 0;
  for (int i = 0; i < 20000; ++i) sink = sink + sfe::sequential_sum(ud(rng), 1 << 30);
  if (sfe::sequential_sum(1.0f, 1 << 30) != 16777216.0f) ++bad;
  printf("checks %ld bad %ld\n", checks, bad);
  return bad != 0;
}

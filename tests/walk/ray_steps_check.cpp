// Host check of RayWalk::steps and seek (bonxai_amd/csrc/bxg_walk.h) on both
// sides of the 32-bit limit (kRay32): the steps taken when a walk reaches
// cell k are floor((2k|d| + m) / (2m)) along each axis, the error terms
// k|d| - n m - ceil(m / 2).
//
// usage: ray_steps_check; prints "ok <checks>" or the first mismatch.
#include <cstdio>
#include <random>

#include "bxg_walk.h"

int main() {
  std::mt19937_64 rng(7);
  long checks = 0;
  for (const int64_t m : {1ll, 2ll, 7ll, 32765ll, 32766ll, 32767ll, 32768ll, 32769ll, 65536ll, 1ll << 24}) {
    for (int t = 0; t < 4000; ++t) {
      int64_t d[3] = {m, (int64_t)(rng() % (uint64_t)(m + 1)), (int64_t)(rng() % (uint64_t)(m + 1))};
      if (t % 3 == 0) d[1] = m;
      if (t % 5 == 0) d[2] = 0;
      const int64_t k = t == 0 ? m : (t == 1 ? 1 : (int64_t)(1 + rng() % (uint64_t)m));
      bxg::RayWalk w;
      w.init(5, -9, 100, 5 + (int32_t)d[0], -9 - (int32_t)d[1], 100 + (int32_t)d[2]);
      int32_t n[3];
      w.steps((int32_t)k, n[0], n[1], n[2]);
      w.seek((int32_t)k, (int32_t)k + 1);
      const int32_t c[3] = {w.cx, w.cy, w.cz}, e[3] = {w.ex, w.ey, w.ez};
      const int32_t o[3] = {5, -9, 100}, s[3] = {1, -1, 1};
      for (int a = 0; a < 3; ++a, ++checks) {
        const int64_t want = (2 * k * d[a] + m) / (2 * m);
        if (n[a] != want || c[a] != o[a] + s[a] * want || e[a] != k * d[a] - want * m - (m + 1) / 2) {
          std::printf("mismatch m %lld k %lld d %lld\n", (long long)m, (long long)k, (long long)d[a]);
          return 1;
        }
      }
    }
  }
  std::printf("ok %ld\n", checks);
  return 0;
}

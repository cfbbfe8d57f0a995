// Host check of the walk with 16-bit error terms (RayWalk16,
// bonxai_amd/csrc/bxg_walk.h) against the 32-bit walk (RayWalk): the same runs
// of cells, the same positions after each, for rays up to its limit of kRay32
// cells, whole and from a seek.
//
// usage: ray_walk16_check; prints "ok <runs>" or the first mismatch.
#include <cstdio>
#include <random>

#include "bxg_walk.h"

int main() {
  std::mt19937_64 rng(5);
  long runs = 0;
  for (const int32_t m : {1, 2, 3, 8, 9, 64, 300, 4097, 32766, 32767}) {
    for (int t = 0; t < (m > 2000 ? 120 : 2000); ++t) {
      const uint32_t lb = 1 + (uint32_t)(rng() % 4);
      int32_t o[3], d[3];
      for (int a = 0; a < 3; ++a) {
        o[a] = (int32_t)(rng() % 40001) - 20000;
        d[a] = (int32_t)(rng() % (uint64_t)(2 * m + 1)) - m;
        if (rng() % 5 == 0) d[a] = 0;
        if (rng() % 5 == 0) d[a] = rng() % 2 ? m : -m;  // as long as the longest axis
      }
      d[t % 3] = rng() % 2 ? m : -m;
      bxg::RayWalk w;
      w.init(o[0], o[1], o[2], o[0] + d[0], o[1] + d[1], o[2] + d[2]);
      const int32_t last = m + (int32_t)(rng() % 2);
      const int32_t k0 = rng() % 2 ? 0 : (int32_t)(rng() % (uint64_t)last);
      const int32_t k1 = k0 + 1 + (int32_t)(rng() % (uint64_t)(last - k0));
      if (k0 == 0)
        w.kend = k1;
      else
        w.seek(k0, k1);
      bxg::RayWalk16 v;
      v.init(w, lb);
      while (!w.done()) {
        uint32_t li[bxg::kRun], lv[bxg::kRun];
        const uint32_t n = bxg::collect_cells(w, lb, li), nv = bxg::collect_cells(v, lb, lv);
        ++runs;
        int32_t a[3], b[3];
        w.cell(a[0], a[1], a[2]);
        v.cell(b[0], b[1], b[2]);
        bool same = n == nv && w.k == v.k && w.done() == v.done() && a[0] == b[0] && a[1] == b[1] && a[2] == b[2];
        for (int j = 0; j < bxg::kRun; ++j) same = same && li[j] == lv[j];
        if (!same) {
          std::printf("mismatch m %d lb %u d %d %d %d at cell %d\n", m, lb, d[0], d[1], d[2], w.k);
          return 1;
        }
      }
      if (!v.done()) return 1;
    }
  }
  std::printf("ok %ld\n", runs);
  return 0;
}

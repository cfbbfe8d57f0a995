// Host check of the leaf walk (LeafWalk, bonxai_amd/csrc/bxg_walk.h): the
// leaves of a ray's cells [k0, k1), in order, as root origin and inner cell,
// against the leaves of the cells one by one.
//
// usage: leaf_walk_check; prints "ok <leaves>" or the first mismatch.
#include <cstdio>
#include <random>

#include "bxg_walk.h"

int main() {
  std::mt19937_64 rng(11);
  long leaves = 0;
  for (uint32_t lb = 1; lb <= 4; ++lb) {
    for (uint32_t ib = 1; ib <= 4; ++ib) {
      for (const int32_t m : {0, 1, 2, 7, 40, 300, 3001, 32766, 32767, 32768, 70001, 1 << 24}) {
        for (int t = 0; t < (m > 5000 ? 12 : 200); ++t) {
          int32_t o[3], d[3];
          for (int a = 0; a < 3; ++a) {
            o[a] = (int32_t)(rng() % 4001) - 2000;
            d[a] = (int32_t)(rng() % (uint64_t)(2 * m + 1)) - m;
          }
          d[t % 3] = t & 1 ? m : -m;
          if (t % 5 == 0) d[(t + 1) % 3] = 0;
          if (t % 7 == 0) d[(t + 2) % 3] = d[t % 3];
          if (t % 11 == 0) d[(t + 1) % 3] = m > 0 ? 1 : 0;
          // the whole ray with its end cell, or a part of it (of the longest, 20000 cells)
          const int32_t last = m + 1;
          const bool whole = t < 20 && m < (1 << 20);
          const int32_t k0 = whole ? 0 : (int32_t)(rng() % (uint64_t)last);
          int32_t k1 = whole ? last : k0 + 1 + (int32_t)(rng() % (uint64_t)(last - k0));
          if (m >= 1 << 20 && k1 - k0 > 20000) k1 = k0 + 20000;
          bxg::RayWalk w;
          w.init(o[0], o[1], o[2], o[0] + d[0], o[1] + d[1], o[2] + d[2]);
          if (k0 == 0)
            w.kend = k1;
          else
            w.seek(k0, k1);
          bxg::LeafWalk lw;
          lw.init(w, lb, ib);
          const int32_t lmask = ~((1 << lb) - 1), rmask = ~((1 << (lb + ib)) - 1), im = (1 << ib) - 1;
          int32_t seen[3] = {0x7fffffff, 0, 0};
          for (int32_t k = k0; k < k1; ++k) {
            int32_t c[3];
            for (int a = 0; a < 3; ++a) {  // cell k by the closed form
              const int64_t n = m ? (2 * (int64_t)k * (d[a] < 0 ? -d[a] : d[a]) + m) / (2 * (int64_t)m) : 0;
              c[a] = o[a] + (d[a] < 0 ? -1 : 1) * (int32_t)n;
            }
            if (k > k0 && (c[0] & lmask) == seen[0] && (c[1] & lmask) == seen[1] && (c[2] & lmask) == seen[2]) continue;
            if (k > k0) lw.next();
            for (int a = 0; a < 3; ++a) seen[a] = c[a] & lmask;
            if (!lw.done() && !lw.inside(ib)) lw.enter(lb, ib);
            const uint32_t ci = (uint32_t)(((c[0] >> lb) & im) | (((c[1] >> lb) & im) << ib) | (((c[2] >> lb) & im) << 2 * ib));
            ++leaves;
            if (lw.done() || lw.k != k || !lw.inside(ib) || lw.cell(ib) != ci || lw.rx != (c[0] & rmask) ||
                lw.ry != (c[1] & rmask) || lw.rz != (c[2] & rmask)) {
              std::printf("mismatch lb %u ib %u m %d t %d cell %d\n", lb, ib, m, t, k);
              return 1;
            }
          }
          lw.next();
          if (!lw.done()) {
            std::printf("a leaf too many: lb %u ib %u m %d t %d\n", lb, ib, m, t);
            return 1;
          }
        }
      }
    }
  }
  std::printf("ok %ld\n", leaves);
  return 0;
}

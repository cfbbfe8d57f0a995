// Host check of the tasks of the ray walks (WalkPlan in
// bonxai_amd/csrc/bxg_walk.h): every segment of every batch is walked once, by
// wavefronts that share the work evenly over the XCDs where batches are few.
//
// usage: walk_plan_check; prints "ok <checks>" or the first mismatch.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "bxg_walk.h"

int main() {
  using namespace bxg;
  long checks = 0;
  for (uint32_t nb : {0u, 1u, 2u, 3u, 7u, 8u, 9u, 31u, 63u, 64u, 65u, 100u, 127u, 128u, 129u, 255u, 256u, 300u, 511u,
                      512u, 513u, 1000u, 2000u, 4801u}) {
    for (uint32_t per : {1u, 3u, 4u, 12u, 16u, 33u, 128u, 400u, 2048u}) {  // wavefronts an XCD
      const WalkPlan plan(nb, per * kXcds);
      std::vector<int> done((size_t)nb << plan.lg, 0);
      uint32_t most = 0;
      for (uint32_t xcd = 0; xcd < kXcds; ++xcd)
        for (uint32_t wave = 0; wave < per; ++wave) {
          uint32_t batch, seg, tasks = 0;
          for (uint32_t j = wave; plan.task(j, xcd, batch, seg); j += per) {
            ++tasks;
            if (batch >= nb) continue;
            if (seg >= 1u << plan.lg) {
              std::printf("%u batches, %u wavefronts: segment %u\n", nb, per, seg);
              return 1;
            }
            ++done[((size_t)batch << plan.lg) + seg];
          }
          most = std::max(most, tasks);
        }
      for (size_t i = 0; i < done.size(); ++i, ++checks)
        if (done[i] != 1) {
          std::printf("%u batches, %u wavefronts an XCD: task %zu done %d times\n", nb, per, i, done[i]);
          return 1;
        }
      // a list of fewer batches than 16 an XCD that is cut: one task a wavefront
      if (nb < 16 * kXcds && !plan.whole() && most > 1) {
        std::printf("%u batches, %u wavefronts an XCD: %u tasks a wavefront\n", nb, per, most);
        return 1;
      }
    }
  }
  std::printf("ok %ld\n", checks);
  return 0;
}

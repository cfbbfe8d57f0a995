// Host check of the parts that a bucket of a bulk cell call is done in
// (bonxai_amd/csrc/bxg_op_parts.h): with tables of the kernel's sizes and
// slots, every cell of a bucket is done in exactly one part that fits, and few
// passes are made over the bucket.  Buckets of `leaves` leaves with `cells`
// cells each; the entries come in an order of their own.
//
// usage: op_parts_check; prints "ok <checks>" or the first mismatch.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "bxg_op_parts.h"

namespace {

uint64_t mix64(uint64_t h) {
  h ^= h >> 33;
  h *= 0xFF51AFD7ED558CCDull;
  h ^= h >> 33;
  h *= 0xC4CEB9FE1A85EC53ull;
  h ^= h >> 33;
  return h;
}

constexpr uint64_t kEmpty = ~0ull;

bool claim(std::vector<uint64_t>& table, uint32_t slot, uint64_t key, uint32_t probes) {
  for (uint32_t p = 0; p < probes; ++p, slot = (slot + 1u) & (uint32_t)(table.size() - 1u)) {
    if (table[slot] == kEmpty) table[slot] = key;
    if (table[slot] == key) return true;
  }
  return false;
}

}  // namespace

int main() {
  using namespace bxg;
  std::mt19937_64 rng(5);
  const struct {
    uint32_t leaves, cells, cell_bits;
    double most;  // passes a bucket on average (a pass for each part, and for each one that had to be halved)
  } cases[] = {
      {54, 18, 9, 1.0},    // clusters
      {300, 4, 9, 1.0},   {1000, 1, 9, 1.5}, {98, 1, 12, 1.0}, {200, 5, 12, 1.0}, {2, 512, 12, 1.0},
      {300, 18, 9, 4.0},   // 5,400 cells: two halves, most of which fit
      {300, 80, 9, 31.0},  // 24,000 cells: 8 to 16 parts
      {4900, 1, 9, 15.0},  // 4 to 8 parts
  };
  long checks = 0;
  for (const auto& k : cases) {
    double passes = 0;
    const int buckets = 40;
    for (int b = 0; b < buckets; ++b) {
      std::vector<uint64_t> cells;
      const uint64_t nb = 2048;  // leaves whose hash ends in the bucket's number
      for (uint32_t l = 0; l < k.leaves;) {
        const uint64_t child = rng() & ((1ull << 26) - 1);
        if ((mix64(child) & (nb - 1)) != (uint64_t)(b * 37 % nb)) continue;
        ++l;
        std::vector<uint32_t> in(1u << k.cell_bits);
        for (uint32_t i = 0; i < in.size(); ++i) in[i] = i;
        std::shuffle(in.begin(), in.end(), rng);
        if (k.cell_bits > kOpUnitLog)  // one unit of the leaf
          for (uint32_t& c : in) c = (c & ((1u << kOpUnitLog) - 1u)) | ((l & 7u) << kOpUnitLog);
        for (uint32_t c = 0; c < k.cells; ++c) cells.push_back((child << k.cell_bits) | in[c]);
      }
      std::sort(cells.begin(), cells.end());
      cells.erase(std::unique(cells.begin(), cells.end()), cells.end());
      std::shuffle(cells.begin(), cells.end(), rng);
      std::vector<int> done(cells.size(), 0);
      OpPart part;
      for (;;) {
        passes += 1;
        std::vector<uint64_t> tl(kOpLeaves, kEmpty), tc(kOpCells, kEmpty);
        std::vector<size_t> mine;
        bool leaves_full = false, cells_full = false;
        for (size_t i = 0; i < cells.size(); ++i) {
          const uint64_t cell = cells[i], unit = cell >> op_unit_log(k.cell_bits / 3), hash = mix64(cell);
          if (!part.whole() && !part.holds(mix64(unit), hash)) continue;
          if (!claim(tl, op_leaf_slot(unit), unit, kOpProbes))
            leaves_full = true;
          else if (!claim(tc, op_cell_slot(cell), cell, kOpProbes))
            cells_full = true;
          mine.push_back(i);
        }
        if (leaves_full || cells_full) {
          if (!part.halve(leaves_full)) {
            std::printf("cannot halve: %u leaves, %u cells\n", k.leaves, k.cells);
            return 1;
          }
          continue;
        }
        for (const size_t i : mine) ++done[i];
        if (!part.next()) break;
      }
      for (size_t i = 0; i < done.size(); ++i, ++checks)
        if (done[i] != 1) {
          std::printf("%u leaves, %u cells: cell %zu done %d times\n", k.leaves, k.cells, i, done[i]);
          return 1;
        }
    }
    if (passes / buckets > k.most) {
      std::printf("%u leaves of %u cells: %.2f passes a bucket\n", k.leaves, k.cells, passes / buckets);
      return 1;
    }
  }
  std::printf("ok %ld\n", checks);
  return 0;
}

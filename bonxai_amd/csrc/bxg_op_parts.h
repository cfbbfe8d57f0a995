// bxg_op_parts.h -- the tables of a bucket of a bulk cell call, and the parts a
// bucket is done in when they cannot hold it.  Plain C++ with no HIP
// dependence, so the same code compiles for the GPU (k_op_buckets) and for the
// host check of tests/test_op_parts.py.
#pragma once

#include <stdint.h>

#if defined(__HIP__)
#define BXG_PARTS_HD __host__ __device__ __forceinline__
#else
#define BXG_PARTS_HD inline
#endif

namespace bxg {

// Slots of a bucket's tables of cells and leaves (powers of two), four times
// and twice a bucket's inputs on average, and how many are looked at for a key
// before a table counts as full.  2M inputs: 3072 slots for cells, four
// workgroups a CU for three, 78 us for 66 (the fuller tables cost more than the
// wavefronts bring); 2048 slots for leaves, with the mask words in the place of
// inputs that are read by then, 58 us, 256 slots beside the mask words 59.
// 2,700 cells fit in most cases with 64 slots looked at, in under half of them
// with 32.
constexpr uint32_t kOpCells = 4096;
constexpr uint32_t kOpLeaves = 2048;
constexpr uint32_t kOpProbes = 64;

// What belongs to one bucket: a leaf, or of a leaf of 16^3 cells a part of 512,
// log2 of its cells.  (As many cells as the table has slots are not done at
// once: 500k inputs in 8 such leaves took 522 us when they were buckets' units.)
constexpr uint32_t kOpUnitLog = 9;
BXG_PARTS_HD uint32_t op_unit_log(uint32_t leaf_bits) { return leaf_bits > 3 ? kOpUnitLog : 3 * leaf_bits; }

// first slot of a cell and of a unit (its leaf's entry among the children, then
// its place in the leaf); a bucket's units are spread by the hash that put them
// there, so a multiplication does
BXG_PARTS_HD uint32_t op_cell_slot(uint64_t cell) {
  return (((uint32_t)cell + (uint32_t)(cell >> 32) * 0x85EBCA6Bu) * 0x9E3779B1u) >> 20;
}
BXG_PARTS_HD uint32_t op_leaf_slot(uint64_t unit) { return ((uint32_t)unit * 0x9E3779B1u) >> 21; }
static_assert(kOpCells == 1u << (32 - 20) && kOpLeaves == 1u << (32 - 21), "slots");

// The part of a bucket that its workgroup holds in its tables: the whole, or
// after a table was full one half after the other, each halved further where it
// has to be.  Where the table of the leaves is full the leaves are divided, by
// their hashes (divided by their cells' hashes, leaves of several cells are in
// nearly every part: with a table of 256 leaves, 300 of 18 cells took 41 passes
// over a bucket, now 3; 20M inputs in 1.2M leaves 18.6 -> 2.6 ms); where only
// that of the cells is, the cells are.
struct OpPart {
  uint32_t leaf_depth = 0, leaf_path = 0, cell_depth = 0, cell_path = 0;
  BXG_PARTS_HD static uint32_t low(uint32_t bits) { return (uint32_t)((1ull << bits) - 1ull); }
  BXG_PARTS_HD bool whole() const { return (leaf_depth | cell_depth) == 0; }
  // the upper halves of the 64-bit hashes (the lower bits give bucket and slot)
  BXG_PARTS_HD bool holds(uint64_t leaf_hash, uint64_t cell_hash) const {
    return ((uint32_t)(leaf_hash >> 32) & low(leaf_depth)) == leaf_path &&
           ((uint32_t)(cell_hash >> 32) & low(cell_depth)) == cell_path;
  }
  // A table was full (`leaves`: that of the leaves): the first half of the part.
  // False where it cannot be halved any further.
  BXG_PARTS_HD bool halve(bool leaves) {
    uint32_t& depth = leaves && cell_depth == 0 ? leaf_depth : cell_depth;
    if (depth == 32) return false;
    ++depth;
    return true;
  }
  // the part after this one; false after the last
  BXG_PARTS_HD bool next() { return step(cell_depth, cell_path) || step(leaf_depth, leaf_path); }
  BXG_PARTS_HD static bool step(uint32_t& depth, uint32_t& path) {
    while (depth && ((path >> (depth - 1u)) & 1u)) path &= ~(1u << --depth);
    if (depth) path |= 1u << (depth - 1u);
    return depth != 0;
  }
};

}  // namespace bxg

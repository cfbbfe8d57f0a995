// bxg_kernels.hip -- gfx950 kernels of the sparse voxel map.
//
// Built with -ffp-contract=off: the scan front end (insertPointCloud's
// max-range clip and posToCoord) must round every FP64 operation exactly as
// the reference's x86-64 double code, which has no fused multiply-add.
//
// Memory-model notes.  Cross-lane races are resolved with agent-scope atomics
// (root-slot claims, leaf claims, endpoint first-index claims, mask bits).
// Reads that only decide whether an atomic is needed are plain loads: a root
// key or a leaf index never changes once published inside a kernel, so a
// stale read can only show the EMPTY word, which sends the lane to the CAS.
// The ray phase writes cell words with plain stores: during that phase every
// update of a cell is the same function of the same prior word (the miss
// update guarded by update_id), so concurrent writers store identical
// values, and a stale read can only return the prior word or the updated
// word, either of which leads to the same final value.
//
// Pointers read out of a map header are cast to the global address space
// (BXG_G) so loads compile to global_load rather than flat_load.
#include "bxg_internal.h"
#include "bxg_op_parts.h"
#include "bxg_walk.h"

#define BXG_G __attribute__((address_space(1)))

namespace bxg {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <class T>
__device__ __forceinline__ T BXG_G* gp(T* p) {
  return (T BXG_G*)p;
}

// --------------------------------------------------------------- atomics

__device__ __forceinline__ uint32_t ld32(const uint32_t* p) {
  return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st32(uint32_t* p, uint32_t v) {
  __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t cas32(uint32_t* p, uint32_t expect, uint32_t desired) {
  __hip_atomic_compare_exchange_strong(gp(p), &expect, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return expect;
}
__device__ __forceinline__ uint64_t cas64(uint64_t* p, uint64_t expect, uint64_t desired) {
  __hip_atomic_compare_exchange_strong(gp(p), &expect, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return expect;
}
__device__ __forceinline__ uint32_t add32(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_add(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t add64(uint64_t* p, uint64_t v) {
  return __hip_atomic_fetch_add(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t or32(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_or(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t or64(uint64_t* p, uint64_t v) {
  return __hip_atomic_fetch_or(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t and64(uint64_t* p, uint64_t v) {
  return __hip_atomic_fetch_and(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t xor64(uint64_t* p, uint64_t v) {
  return __hip_atomic_fetch_xor(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t min32(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_min(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
__device__ __forceinline__ uint64_t lanes_below() { return (1ull << lane_id()) - 1ull; }

// Minimum over the 64 lanes of a wavefront, every lane active: DPP moves
// within quads (quad_perm [1,0,3,2], [2,3,0,1]) and rows (row_ror 4, 8), then
// row_bcast 15 into rows 1 and 3 and row_bcast 31 into rows 2 and 3, so that
// lane 63 holds the minimum; no LDS round trips.  The value kept where a move
// writes nothing is the operation's identity, so that the compiler makes the
// move a modifier of the operation.
__device__ __forceinline__ int32_t wave_min(int32_t v) {
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0xB1, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0x4E, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0x124, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0x128, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0x142, 0xA, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// bitwise or over the 64 lanes of a wavefront, every lane active (the steps
// of wave_min)
__device__ __forceinline__ uint32_t wave_or32(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint64_t wave_or(uint64_t v) {
  return (uint64_t)wave_or32((uint32_t)v) | ((uint64_t)wave_or32((uint32_t)(v >> 32)) << 32);
}

// value of lane l (the same l in every lane), 64 bits
__device__ __forceinline__ uint64_t lane_value(uint64_t v, uint32_t l) {
  return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)l) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)l) << 32);
}

// Bump allocation from per-map counters, aggregated over a wavefront: the
// active lanes with pred set are grouped by counter address (lanes of one
// wavefront usually serve one map), each group takes one atomic add of its
// size, and each lane gets base + its rank in the group.  Every active lane
// must call it (it is a wavefront collective); the result is meaningful only
// where pred is set.
__device__ __forceinline__ uint32_t wave_bump(uint32_t* counter, bool pred) {
  uint64_t pending = __ballot(pred);
  uint32_t mine = 0;
  while (pending) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const unsigned long long lc = __shfl((unsigned long long)counter, leader);
    const uint64_t same = __ballot(pred && (unsigned long long)counter == lc);
    uint32_t base = 0;
    if ((int)lane_id() == leader) base = add32((uint32_t*)lc, (uint32_t)__popcll(same));
    base = __shfl(base, leader);
    if ((same >> lane_id()) & 1ull) mine = base + (uint32_t)__popcll(same & lanes_below());
    pending &= ~same;
  }
  return mine;
}

// The lowest lane of this lane's run: the maximal block of consecutive lanes
// that all have `on` set and equal (k1, k2).  Lanes of a wavefront that share
// a table entry and sit side by side let that lane do the entry's atomics
// for all of them.  Every lane must call it; the result means something only
// where `on` is set.
__device__ __forceinline__ int run_leader(bool on, uint64_t k1, uint32_t k2) {
  const uint32_t lane = lane_id();
  // the previous lane's keys: DPP wave_shr:1 (lane i reads lane i - 1; lane
  // 0's value is not used), no LDS round trip
  const uint32_t k1lo = (uint32_t)k1, k1hi = (uint32_t)(k1 >> 32);
  const uint32_t p1lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k1lo, 0x138, 0xF, 0xF, false);
  const uint32_t p1hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k1hi, 0x138, 0xF, 0xF, false);
  const uint64_t p1 = ((uint64_t)p1hi << 32) | p1lo;
  const uint32_t p2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k2, 0x138, 0xF, 0xF, false);
  const uint64_t onmask = __ballot(on);
  const bool prev_on = lane > 0 && ((onmask >> (lane - 1)) & 1ull);
  const bool start = on && !(prev_on && p1 == k1 && p2 == k2);
  const uint64_t upto = __ballot(start) & (~0ull >> (63u - lane));
  return upto ? 63 - __clzll(upto) : (int)lane;
}

// ------------------------------------------------------------ map view

// A register copy of a map header with global-address-space pointers.
struct MapView {
  uint64_t BXG_G* root_keys;
  uint32_t BXG_G* children;
  uint64_t BXG_G* masks;
  uint8_t BXG_G* cells;
  uint8_t BXG_G* touched;
  int4* origin;  // HIP vector types keep the generic address space
  MapCounters* ctr;
  double inv_res;
  uint32_t ib, lb, log2n, isz, lsz, lw, vb, flags;
  uint64_t BXG_G* have;
  uint64_t BXG_G* want;
  uint32_t root_mask, max_probe, leaf_cap;
  int32_t miss, hit, cmin, cmax, thr;
};

__device__ __forceinline__ MapView load_view(const MapDev* p) {
  const MapDev BXG_G* q = (const MapDev BXG_G*)p;
  MapView v;
  v.root_keys = gp(q->root_keys);
  v.children = gp(q->children);
  v.masks = gp(q->leaf_masks);
  v.cells = gp(q->cells);
  v.touched = gp(q->touched);
  v.origin = q->leaf_origin;
  v.ctr = q->ctr;
  v.inv_res = q->inv_res;
  v.ib = q->inner_bits;
  v.lb = q->leaf_bits;
  v.log2n = q->log2n;
  v.isz = q->inner_size;
  v.lsz = q->leaf_size;
  v.lw = q->leaf_words;
  v.vb = q->value_bytes;
  v.flags = q->flags;
  v.have = gp((uint64_t*)q->leaf_have);
  v.want = gp((uint64_t*)q->leaf_want);
  v.root_mask = q->root_mask;
  v.max_probe = q->max_probe;
  v.leaf_cap = q->leaf_cap;
  v.miss = q->opt_miss;
  v.hit = q->opt_hit;
  v.cmin = q->opt_cmin;
  v.cmax = q->opt_cmax;
  v.thr = q->opt_thr;
  return v;
}

// A map header read through scalar loads: p is the same in every lane of the
// wavefront (a header changes only between kernels).
#define BXG_C __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ T* uniform_ptr(T* p) {
  const uint64_t a = (uint64_t)p;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
  return (T*)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int32_t uniform_i32(const int32_t* p) {
  return *(const int32_t BXG_C*)uniform_ptr(p);
}
__device__ __forceinline__ MapView uniform_view(const MapDev* p) {
  const MapDev BXG_C* q = (const MapDev BXG_C*)uniform_ptr(p);
  MapView v;
  v.root_keys = gp((uint64_t*)q->root_keys);
  v.children = gp((uint32_t*)q->children);
  v.masks = gp((uint64_t*)q->leaf_masks);
  v.cells = gp((uint8_t*)q->cells);
  v.touched = gp((uint8_t*)q->touched);
  v.origin = q->leaf_origin;
  v.ctr = q->ctr;
  v.inv_res = q->inv_res;
  v.ib = q->inner_bits;
  v.lb = q->leaf_bits;
  v.log2n = q->log2n;
  v.isz = q->inner_size;
  v.lsz = q->leaf_size;
  v.lw = q->leaf_words;
  v.vb = q->value_bytes;
  v.flags = q->flags;
  v.have = gp((uint64_t*)q->leaf_have);
  v.want = gp((uint64_t*)q->leaf_want);
  v.root_mask = q->root_mask;
  v.max_probe = q->max_probe;
  v.leaf_cap = q->leaf_cap;
  v.miss = q->opt_miss;
  v.hit = q->opt_hit;
  v.cmin = q->opt_cmin;
  v.cmax = q->opt_cmax;
  v.thr = q->opt_thr;
  return v;
}

// counter words read at kernel start (written by earlier kernels)
__device__ __forceinline__ uint32_t map_status(const MapView& m) { return *gp(&m.ctr->status); }
__device__ __forceinline__ int32_t map_cur(const MapView& m) { return *gp(&m.ctr->cur); }

constexpr uint32_t kFatal = kStOutOfPool | kStRootFull | kStCoordRange | kStScratchFull;

// ---------------------------------------------------------- directory

__device__ __forceinline__ uint32_t root_hash(uint64_t key, uint32_t mask) {
  return (uint32_t)mix64(key) & mask;
}

// Find-or-insert of a root key (lock-free CAS insert, linear probing).
// Returns the slot, or -1 (and sets kStRootFull) after max_probe probes;
// `inserted` tells whether this lane's CAS created it (the caller counts it).
__device__ int32_t root_probe(const MapView& m, uint64_t key, bool& inserted) {
  uint32_t h = root_hash(key, m.root_mask);
  inserted = false;
  for (uint32_t p = 0; p < m.max_probe; ++p) {
    uint64_t k = m.root_keys[h];
    if (k == kEmptyKey) {
      k = cas64((uint64_t*)&m.root_keys[h], kEmptyKey, key);
      if (k == kEmptyKey) {
        inserted = true;
        return (int32_t)h;
      }
    }
    if (k == key) return (int32_t)h;
    h = (h + 1) & m.root_mask;
  }
  or32(&m.ctr->status, kStRootFull);
  return -1;
}

// root_probe with the roots a wavefront inserts counted by one atomic per
// map (wave_bump), so every active lane must call it.
__device__ int32_t root_insert(const MapView& m, uint64_t key) {
  bool inserted;
  const int32_t slot = root_probe(m, key, inserted);
  wave_bump(&m.ctr->root_count, inserted);
  return slot;
}

// Lookup of a root key in a phase where no insert runs concurrently.
__device__ __forceinline__ int32_t root_find(const MapView& m, uint64_t key) {
  uint32_t h = root_hash(key, m.root_mask);
  for (uint32_t p = 0; p <= m.root_mask; ++p) {
    const uint64_t k = m.root_keys[h];
    if (k == key) return (int32_t)h;
    if (k == kEmptyKey) return -1;
    h = (h + 1) & m.root_mask;
  }
  return -1;
}

// Claim of the inner-grid entry *cp for a new leaf: true if this lane moved
// it from EMPTY to PENDING; otherwise `seen` is the entry as found (a leaf
// index, or PENDING while another lane creates the leaf).
__device__ __forceinline__ bool leaf_claim(uint32_t* cp, uint32_t& seen) {
  uint32_t v = *gp(cp);
  if (v == kEmptyChild) v = cas32(cp, kEmptyChild, kPendingChild);
  seen = v;
  return v == kEmptyChild;
}

// Leaf indices for the lanes that claimed an entry (allocateLeafGrid and
// GridBlockAllocator::allocateBlock, bonxai.hpp:572-586 and
// grid_allocator.hpp:94-123): one wavefront-aggregated bump of the map's
// leaf counter per wavefront and map, then each claimer writes its leaf's
// origin and publishes the index in the entry.  A claimer past the pool's
// capacity puts the entry back to EMPTY and flags the map (the host grows the
// pool and runs the call again).  Every active lane must call it; returns the
// new index, or EMPTY on failure, where `claimed` is set.
__device__ __forceinline__ uint32_t leaf_publish(const MapView& m, bool claimed, uint32_t* cp,
                                                 uint32_t slot, int32_t lx, int32_t ly, int32_t lz) {
  const uint32_t idx = wave_bump(&m.ctr->leaf_count, claimed);
  if (!claimed) return kEmptyChild;
  if (idx >= m.leaf_cap) {
    st32(cp, kEmptyChild);
    or32(&m.ctr->status, kStOutOfPool);
    return kEmptyChild;
  }
  m.origin[idx] = make_int4(lx, ly, lz, (int32_t)slot);
  st32(cp, idx);
  return idx;
}

// Make sure leaf `ci` of root `slot` exists (a wavefront collective, through
// leaf_publish).  Returns the child word as seen: a leaf index, PENDING while
// another lane creates it, or EMPTY when the pool ran out.
__device__ __forceinline__ uint32_t leaf_request(const MapView& m, uint32_t slot, uint32_t ci,
                                                 int32_t lx, int32_t ly, int32_t lz) {
  uint32_t* cp = (uint32_t*)&m.children[(uint64_t)slot * m.isz + ci];
  uint32_t seen;
  const bool won = leaf_claim(cp, seen);
  const uint32_t idx = leaf_publish(m, won, cp, slot, lx, ly, lz);
  return won ? idx : seen;
}

// leaf index holding coordinate c, or kNone (read-only phases)
__device__ __forceinline__ uint32_t find_leaf(const MapView& m, int32_t x, int32_t y, int32_t z) {
  uint64_t key;
  if (!pack_root(x, y, z, m.log2n, &key)) return kNone;
  const int32_t s = root_find(m, key);
  if (s < 0) return kNone;
  const uint32_t c = m.children[(uint64_t)s * m.isz + inner_index(x, y, z, m.lb, m.ib)];
  return c >= kPendingChild ? kNone : c;
}

// The root slot of the last root a walk visited.
struct RootCache {
  int32_t rx, ry, rz, slot;
  bool valid;
  // fields set, so that the cache test below may read them without branches
  __device__ __forceinline__ void reset() {
    rx = ry = rz = 0;
    slot = -1;
    valid = false;
  }
};

// slot of the root holding (x, y, z): looked up (kInsert false) or created
// (kInsert true), cached while the walk stays in the root
template <bool kInsert>
__device__ __forceinline__ int32_t root_slot(const MapView& m, RootCache& rc, int32_t x, int32_t y,
                                             int32_t z) {
  const int32_t rmask = ~((1 << m.log2n) - 1);
  const int32_t rx = x & rmask, ry = y & rmask, rz = z & rmask;
  if (!rc.valid | (((rx ^ rc.rx) | (ry ^ rc.ry) | (rz ^ rc.rz)) != 0)) {
    uint64_t key;
    int32_t s = -1;
    if (pack_root(x, y, z, m.log2n, &key)) s = kInsert ? root_insert(m, key) : root_find(m, key);
    rc.rx = rx;
    rc.ry = ry;
    rc.rz = rz;
    rc.slot = s;
    rc.valid = true;
  }
  return rc.slot;
}

// ------------------------------------------------------- cell update

// signed 4-bit update_id and 28-bit log-odds of a CellT word
__device__ __forceinline__ int32_t cell_id(uint32_t w) { return ((int32_t)(w << 28)) >> 28; }
__device__ __forceinline__ int32_t cell_p(uint32_t w) { return ((int32_t)w) >> 4; }

// probability_log = min(p + hit, clamp_max) or max(p + miss, clamp_min),
// update_id = cur: addHitPoint, addMissPoint and the clearPoint lambda
// (probabilistic_map.cpp:30-41, 43-54, 81-89); the sum wraps like the
// reference's int arithmetic and the store keeps the low 28 bits like its
// 28-bit bit-field.
__device__ __forceinline__ uint32_t cell_hit(uint32_t w, int32_t hit, int32_t cmax, int32_t cur) {
  int32_t p = (int32_t)((uint32_t)cell_p(w) + (uint32_t)hit);
  p = p < cmax ? p : cmax;
  return ((uint32_t)p << 4) | ((uint32_t)cur & 0xFu);
}
__device__ __forceinline__ uint32_t cell_miss(uint32_t w, int32_t miss, int32_t cmin, int32_t cur) {
  int32_t p = (int32_t)((uint32_t)cell_p(w) + (uint32_t)miss);
  p = p > cmin ? p : cmin;
  return ((uint32_t)p << 4) | ((uint32_t)cur & 0xFu);
}

// ------------------------------------------------------------- rays

// The cell walk of a ray (RayWalk, collect_cells) is in bxg_walk.h, shared
// with the host check of the walk.
template <class Walk>
__device__ __forceinline__ uint32_t collect_run(const MapView& m, Walk& w, uint32_t li[kRun]) {
  return collect_cells(w, m.lb, li);
}

// Allocation pass, one step of a ray: the root of its current leaf (created
// if missing) and the ray's next leaves of that root, up to kLeafRun, as bits
// of the root's inner cells.  One load of `known` tells which of them exist
// (the have bits; in a map empty at the scan's start the want bits: those put
// down already); the others are put down in the root's want bits, and
// k_scan_new_entries creates them.  (Leaves created by the rays themselves, a
// claim each and one bump of the map's leaf counter a wavefront and step,
// were bound by the counter, about 6 ns an atomic: 97 us for a LiDAR scan
// that adds 38k leaves to a map, now 40; and a first scan's rays, creating
// leaves and marking cells in one walk, took 465 us, now 60 + 230.)
constexpr int kLeafRun = 8;
constexpr int32_t kNoRoot = -2;  // the root is not looked up yet
__device__ __forceinline__ void leaves_step(const MapView& m, LeafWalk& lw, int32_t& slot,
                                            const uint64_t BXG_G* known, bool go) {
  uint64_t miss = 0;
  uint32_t e = 0;  // word of the directory (at most 2^24 roots of 64 words)
  if (go) {
    if (!lw.inside(m.ib)) {
      lw.enter(m.lb, m.ib);
      slot = kNoRoot;
    }
    if (slot == kNoRoot) {
      uint64_t key;
      slot = pack_root(lw.rx, lw.ry, lw.rz, m.log2n, &key) ? root_insert(m, key) : -1;
    }
    const uint32_t ci = lw.cell(m.ib);
    const uint32_t word = ci >> 6;
    const uint32_t mask = LeafWalk::inside_mask(m.ib) | LeafWalk::word_mask(m.ib);
    const uint32_t here = lw.p & mask;  // this root, this word
    uint64_t bits = 1ull << (ci & 63u);
    lw.next();
#pragma unroll
    for (int j = 1; j < kLeafRun; ++j) {
      if (lw.done() | ((lw.p & mask) != here)) break;
      bits |= 1ull << (lw.p & LeafWalk::kBit);
      lw.next();
    }
    if (slot >= 0) {  // else the root directory is full: the call fails
      e = (uint32_t)slot * entry_words(m.isz) + word;
      miss = bits & ~known[e];
    }
  }
  if (__ballot(miss != 0) == 0) return;
  // Fewer atomics: a lane leaves the bits that the lane before it puts down,
  // and the lanes of the first few words of the wavefront go together on one
  // of them (near the sensor all 64 rays cross one root: a 100k-point room 37
  // us, 120 us without; grouping every word costs more than its atomics where
  // the rays have spread).
  const uint32_t plo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)miss, 0x138, 0xF, 0xF, false);
  const uint32_t phi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(miss >> 32), 0x138, 0xF, 0xF, false);
  const uint32_t pe = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x138, 0xF, 0xF, false);
  uint64_t put = miss;
  if (lane_id() > 0 && pe == e) put &= ~(((uint64_t)phi << 32) | plo);
  uint64_t pending = __ballot(put != 0);
  for (int g = 0; g < 4 && pending; ++g) {
    const uint32_t l = (uint32_t)__ffsll((unsigned long long)pending) - 1u;
    const bool mine = put != 0 && e == (uint32_t)__builtin_amdgcn_readlane((int)e, (int)l);
    pending &= ~__ballot(mine);
    const uint64_t all = wave_or(mine ? put : 0ull);
    if (mine) put = lane_id() == l ? all : 0ull;
  }
  if (put) or64((uint64_t*)&m.want[e], put);
}

// leaf index of the walk's current cell (read-only phases)
template <class Walk>
__device__ __forceinline__ uint32_t walk_leaf(const MapView& m, const Walk& w, RootCache& rc) {
  int32_t x, y, z;
  w.cell(x, y, z);
  const int32_t slot = root_slot<false>(m, rc, x, y, z);
  if (slot < 0) return kNone;
  const uint32_t c = m.children[(uint64_t)slot * m.isz + inner_index(x, y, z, m.lb, m.ib)];
  return c >= kPendingChild ? kNone : c;
}

// One leaf of a ray, update pass: the cells of the ray in the current leaf
// (up to kRun) are loaded together, then each takes the miss update unless
// its update_id already equals cur.  Returns the cells written (counted
// form: exact, by CAS).
//
// next_leaf is the leaf of the walk's current cell on entry; on return it is the
// leaf of the next run (looked up before this run's cells are loaded, so the
// two memory round trips overlap).
//
// Leaves at or above `lbase` were created by the running scan: each of their
// cells was off (zero) before it, and the ray update of such a cell gives the
// same word whichever ray gets there first, cell_miss(0).  So a run in a new
// leaf only marks its cells in the leaf's touched bytes (plain byte stores of
// the miss mark, every writer agreeing; no read, no atomic), and k_scan_new_leaves writes
// the leaf's cells and mask words from those bytes after the scan's endpoints
// are marked.  In older leaves each cell is read, updated unless its
// update_id is cur, and the cells turned on set their mask bits with atomicOrs.
template <bool kCount, class Walk>
__device__ __forceinline__ uint32_t apply_step(const MapView& m, Walk& w, RootCache& rc,
                                               int32_t cur, uint32_t lbase, uint32_t mark,
                                               uint32_t& next_leaf) {
  const uint32_t leaf = next_leaf;
  uint32_t li[kRun];
  const uint32_t n = collect_run(m, w, li);
  next_leaf = w.done() ? kNone : walk_leaf(m, w, rc);
  if (leaf == kNone) return 0;
  if (leaf >= lbase) {
    uint8_t BXG_G* tb = m.touched + (uint64_t)leaf * m.lsz;
    uint32_t nupd = 0;
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
      if ((uint32_t)j < n) {
        if (kCount) {
          // exact first marks: a CAS on the byte's aligned word
          const uint32_t sh = (li[j] & 3u) * 8u;
          uint32_t* wp = (uint32_t*)(tb + (li[j] & ~3u));
          for (uint32_t old = ld32(wp); ((old >> sh) & 0xFFu) != mark;) {
            const uint32_t seen = cas32(wp, old, (old & ~(0xFFu << sh)) | (mark << sh));
            nupd += seen == old ? 1u : 0u;
            if (seen == old) break;
            old = seen;
          }
        } else {
          tb[li[j]] = (uint8_t)mark;
        }
      }
    }
    return nupd;
  }
  uint32_t BXG_G* base = (uint32_t BXG_G*)m.cells + (uint64_t)leaf * m.lsz;
  uint32_t v[kRun];
#pragma unroll
  for (int j = 0; j < kRun; ++j)
    v[j] = base[li[j]];  // slots j >= n re-read the run's first cell
  uint32_t nupd = 0;
  // Mask bits of the cells turned on, gathered per mask word (a plane of the
  // leaf: a ray's cells in it seldom change words more than once), so that a
  // run takes one or two device-wide atomics instead of up to 8: they bound
  // the update pass of scans that turn many cells on (LiDAR scans 1 m apart
  // at 50 m: 357 -> 275 us a scan with 256-thread workgroups)
  uint64_t BXG_G* mw = m.masks + (uint64_t)leaf * m.lw;
  uint32_t word = 0;
  uint64_t bits = 0;
#pragma unroll
  for (int j = 0; j < kRun; ++j) {
    const bool upd = ((uint32_t)j < n) & (cell_id(v[j]) != cur);  // one branch, not two
    if (upd) {
      uint32_t old = v[j];
      if (kCount) {
        for (;;) {
          const uint32_t seen = cas32((uint32_t*)&base[li[j]], old, cell_miss(old, m.miss, m.cmin, cur));
          if (seen == old) {
            ++nupd;
            break;
          }
          old = seen;
          if (cell_id(old) == cur) break;
        }
      } else {
        base[li[j]] = cell_miss(old, m.miss, m.cmin, cur);
      }
      if (old == 0) {
        if (bits != 0 && (li[j] >> 6) != word) {
          or64((uint64_t*)&mw[word], bits);
          bits = 0;
        }
        word = li[j] >> 6;
        bits |= 1ull << (li[j] & 63u);
      }
    }
  }
  if (bits) or64((uint64_t*)&mw[word], bits);
  return nupd;
}

// --------------------------------------------------------- scan phases

__device__ __forceinline__ uint32_t find_scan(const ScanDesc* __restrict__ sd, uint32_t nscans,
                                              uint64_t gi) {
  uint32_t lo = 0, hi = nscans;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (sd[mid].pt_off <= gi)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint64_t ep_key(uint32_t tag, uint32_t slot, uint32_t ci, uint32_t li) {
  return ((uint64_t)tag << 48) | ((uint64_t)slot << 24) | ((uint64_t)ci << 12) | (uint64_t)li;
}

// Phase 0 (per scan): the leaf count at the start of the scan, so that later
// phases can tell the leaves the scan creates from older ones, and the scan's
// update id.
__device__ __forceinline__ void scan_begin(uint32_t nscans, const ScanDesc* sd) {
  for (uint32_t s = threadIdx.x; s < nscans; s += blockDim.x) {
    const MapDev BXG_G* m = gp((const MapDev*)sd[s].map);
    MapCounters BXG_G* ctr = gp(m->ctr);
    ctr->leaf_base = min(ctr->leaf_count, m->leaf_cap);
    ctr->scan_cur = ctr->cur;
  }
}
__global__ void k_scan_begin(const BatchHdr* __restrict__ hdr, const ScanDesc* __restrict__ sd) {
  scan_begin(hdr->nscans, sd);
}

// The same for a call whose batch header and up to kN scan descriptors come
// as kernel arguments, written here into the device buffers that the later
// kernels read: no copy to the device before the call (two small copies and
// the waits around them cost about 35 us at the head of a call).  kN 16 fits
// the 4 KB of a launch's arguments.  With reset_stats (counted calls) the
// maps' scan statistics are cleared.
template <uint32_t kN>
struct ScanArgs {
  ScanDesc d[kN];
};
constexpr uint32_t kMostArgs = 16;
static_assert(sizeof(ScanArgs<kMostArgs>) + sizeof(ScanScratch) + 64 <= 4096, "kernel arguments");
template <uint32_t kN>
__device__ __forceinline__ void scan_begin_args(const BatchHdr& hdr, const ScanArgs<kN>& a, BatchHdr* hdr_out,
                                                ScanDesc* desc_out, uint32_t reset_stats) {
  if (threadIdx.x == 0) *hdr_out = hdr;
  const uint32_t* src = reinterpret_cast<const uint32_t*>(&a);
  uint32_t* dst = reinterpret_cast<uint32_t*>(desc_out);
  const uint32_t words = hdr.nscans * (uint32_t)(sizeof(ScanDesc) / 4);
  for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) dst[i] = src[i];
  if (reset_stats && threadIdx.x < hdr.nscans) {
    MapCounters* ctr = gp((const MapDev*)a.d[threadIdx.x].map)->ctr;
    ctr->stat_rays = 0;
    ctr->stat_ray_updates = 0;
    ctr->stat_ray_visits = 0;
  }
  scan_begin(hdr.nscans, a.d);
}
__global__ void k_scan_begin_args(BatchHdr hdr, ScanArgs<kMostArgs> a, BatchHdr* __restrict__ hdr_out,
                                  ScanDesc* __restrict__ desc_out, uint32_t reset_stats) {
  scan_begin_args(hdr, a, hdr_out, desc_out, reset_stats);
}

// Phase 1 (per point): max-range clip and posToCoord in FP64
// (probabilistic_map.hpp:144-157, bonxai.hpp:404-410), root and leaf of the
// endpoint created, pre-scan update_id test, and the first-index claim of
// the endpoint voxel among the points whose voxel is to be updated.
// kOne: a call of one scan, whose header sits in scalar registers.
template <bool kOne>
__device__ __forceinline__ void classify_points(uint64_t total, uint32_t nscans, const ScanDesc* sd,
                                                const ScanScratch& sc) {
  const uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gi - lane_id() >= total) return;  // the whole wavefront lies past the last point
  // Every lane of a live wavefront stays to the end: the root, leaf and
  // endpoint claims below are wavefront collectives.
  const bool live = gi < total;
  // the scan of the wavefront's first point, searched once with uniform
  // (scalar) loads; lanes past a scan boundary step forward from it
  uint32_t s = 0;
  if (!kOne) {
    const uint64_t g0 = (uint64_t)blockIdx.x * blockDim.x +
                        ((uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) << 6);
    s = find_scan(sd, nscans, g0);
    if (live)
      while (s + 1 < nscans && sd[s + 1].pt_off <= gi) ++s;
    else
      s = 0u;
  }
  const ScanDesc& d = sd[s];
  const MapView m = kOne ? uniform_view(d.map) : load_view(d.map);
  int4 rec = make_int4(0, 0, 0, (int32_t)(s << 16));
  bool valid = false;
  bool clipped = false;
  int32_t ex = 0, ey = 0, ez = 0;
  uint32_t flags = kRecValid;
  if (live) {
    const uint64_t i = gi - d.pt_off;
    double tx, ty, tz;
    bool finite = true;
    const uint8_t BXG_G* pb = gp((const uint8_t*)d.points) + i * d.stride;
    if (d.flags & kScanF64) {
      const double BXG_G* p = (const double BXG_G*)pb;
      tx = p[0];
      ty = p[1];
      tz = p[2];
    } else {
      const float BXG_G* p = (const float BXG_G*)pb;
      float x = p[0], y = p[1], z = p[2];
      if (d.flags & kScanTransform) {
        // bonxai_server.cpp:147-153 drops points with a non-finite coordinate
        finite = __builtin_isfinite(x) && __builtin_isfinite(y) && __builtin_isfinite(z);
        // pcl::transformPointCloud in float (bonxai_server.cpp:166-170), no contraction
        const float* t = d.tf;
        const float nx = t[0] * x + (t[1] * y + (t[2] * z + t[3]));
        const float ny = t[4] * x + (t[5] * y + (t[6] * z + t[7]));
        const float nz = t[8] * x + (t[9] * y + (t[10] * z + t[11]));
        x = nx;
        y = ny;
        z = nz;
      }
      tx = (double)x;
      ty = (double)y;
      tz = (double)z;
    }
    if (finite) {
      const double vx = tx - d.fx, vy = ty - d.fy, vz = tz - d.fz;
      const double sq = (vx * vx + vy * vy) + vz * vz;
      double qx = tx, qy = ty, qz = tz;
      if (d.flags & (kScanForceHit | kScanForceMiss)) {
        if (d.flags & kScanForceHit) flags |= kRecHit;
      } else if (sq >= d.r2) {
        clipped = true;
        const double sr = __builtin_sqrt(sq);
        qx = d.fx + ((vx / sr) * d.max_range);
        qy = d.fy + ((vy / sr) * d.max_range);
        qz = d.fz + ((vz / sr) * d.max_range);
      } else {
        flags |= kRecHit;
      }
      const double ax = __builtin_floor(qx * m.inv_res);
      const double ay = __builtin_floor(qy * m.inv_res);
      const double az = __builtin_floor(qz * m.inv_res);
      const double lim = (double)(1 << (20 + m.log2n));
      if (ax >= -lim && ax < lim && ay >= -lim && ay < lim && az >= -lim && az < lim) {
        valid = true;
        ex = (int32_t)ax;
        ey = (int32_t)ay;
        ez = (int32_t)az;
      } else {
        or32(&m.ctr->status, kStCoordRange);
      }
    }
  }
  // The endpoint's root (created if missing), then its leaf (looked up),
  // then its first-index claim.  Neighbouring points of a scan usually share
  // a root and often a voxel, and neighbouring points sit in neighbouring
  // lanes: each run of lanes with the same key does the table work once, on
  // its lowest lane (run_leader), and the others take the result from it.
  uint64_t rkey = 0;
  if (valid) pack_root(ex, ey, ez, m.log2n, &rkey);
  const int rl = run_leader(valid, rkey, s);
  int32_t slot = -1;
  bool rnew = false;
  // the runs of one root that looks missing go together too: in a new map
  // every wavefront meets the same few missing roots, and each claim is an
  // atomic (64 first scans: 572 -> 523 us, a 100k-point room 43 -> 38 us)
  const bool leads = valid && rl == (int)lane_id();
  const bool missing = leads && m.root_keys[root_hash(rkey, m.root_mask)] == kEmptyKey;
  int lead = rl;
  for (uint64_t pending = __ballot(missing); pending;) {
    const uint32_t l = (uint32_t)__ffsll((unsigned long long)pending) - 1u;
    const bool same = missing && rkey == lane_value(rkey, l) &&
                      s == (uint32_t)__builtin_amdgcn_readlane((int)s, (int)l);
    if (same) lead = (int)l;
    pending &= ~__ballot(same);
  }
  if (leads && lead == (int)lane_id()) slot = root_probe(m, rkey, rnew);
  wave_bump(&m.ctr->root_count, rnew);
  slot = __shfl(slot, lead);  // of a run's leader: from its group's lane
  slot = __shfl(slot, rl);
  if (valid && slot < 0) {
    rec = make_int4(ex, ey, ez, (int32_t)(s << 16));
    valid = false;
  }
  uint32_t ci = 0, li = 0;
  if (valid) {
    ci = inner_index(ex, ey, ez, m.lb, m.ib);
    li = leaf_index(ex, ey, ez, m.lb);
  }
  // the endpoint's leaf as it was before the scan (the leaf pass creates the
  // winners' endpoint leaves; nothing creates leaves in this kernel): a
  // missing leaf means a cell with update_id 0, never cur
  const uint32_t leaf = valid ? *gp(&m.children[(uint64_t)slot * m.isz + ci]) : kEmptyChild;
  bool marked = valid;
  if (valid && leaf < kPendingChild) {
    const uint32_t w = ((const uint32_t BXG_G*)m.cells)[(uint64_t)leaf * m.lsz + li];
    marked = cell_id(w) != map_cur(m);
  }
  // first point of each voxel: lanes are in point order, so a run's lowest
  // lane holds its smallest index, the one the endpoint table keeps
  const uint64_t key = marked ? ep_key(d.tag, (uint32_t)slot, ci, li) : 0ull;
  const int el = run_leader(marked, key, 0u);
  uint32_t tp = kNone;
  if (marked && el == (int)lane_id()) {
    uint32_t h = (uint32_t)mix64(key) & sc.ep_mask;
    for (uint32_t p = 0; p <= sc.ep_mask; ++p) {
      // the slot's key and first index in one load; the index only falls, so
      // one as low already needs no atomic (a depth frame has tens of points
      // a voxel: 41 -> 31 us)
      const u32x4 slot4 = *(const u32x4 BXG_G*)gp(&sc.ep[h]);
      uint64_t k = ((uint64_t)slot4.y << 32) | slot4.x;
      if (k == kEmptyKey) {
        k = cas64(&sc.ep[h].key, kEmptyKey, key);
        if (k == kEmptyKey) k = key;
      }
      if (k == key) {
        if (slot4.z > (uint32_t)gi) min32(&sc.ep[h].first, (uint32_t)gi);
        tp = h;
        break;
      }
      h = (h + 1) & sc.ep_mask;
    }
  }
  tp = __shfl(tp, el);
  if (marked) {
    if (tp == kNone) {
      or32(&m.ctr->status, kStScratchFull);
    } else {
      flags |= kRecMarked;
      sc.tpos[gi] = tp;
    }
  }
  if (valid) rec = make_int4(ex, ey, ez, (int32_t)(flags | (s << 16)));
  if (live) sc.rec[gi] = rec;
  // points clipped at the max range, per scan, counted on one wavefront in
  // 16 (one add per scan of the wavefront; the words share two cache lines,
  // and an add from every wavefront measured 0.5 ms a 6.9 M-point frame):
  // k_scan_winners orders the rays by length only in scans that mix such
  // rays with returns
  uint64_t pend = ((gi >> 6) & 15u) == 0 ? __ballot(clipped) : 0ull;
  while (pend) {
    const int leader = __ffsll((unsigned long long)pend) - 1;
    const uint32_t ls = (uint32_t)__shfl((int)s, leader);
    const uint64_t same = __ballot(clipped && s == ls);
    if ((int)lane_id() == leader) add32(&sc.counters[kClipWords + (ls & 63u)], (uint32_t)__popcll(same));
    pend &= ~same;
  }
}

__global__ void __launch_bounds__(256) k_scan_classify(const BatchHdr* __restrict__ hdr,
                                                       const ScanDesc* __restrict__ sd,
                                                       ScanScratch sc) {
  classify_points<false>(hdr->total, hdr->nscans, sd, sc);
}

// Phases 0 and 1 of a call of one scan in one kernel, the scan as an
// argument: the first workgroup also starts the scan (the points do not need
// what it writes).  A launch saved, about 5 us a call.
__global__ void __launch_bounds__(256) k_scan_classify_one(BatchHdr hdr, ScanArgs<1> a,
                                                           BatchHdr* __restrict__ hdr_out,
                                                           ScanDesc* __restrict__ desc_out, ScanScratch sc,
                                                           uint32_t reset_stats) {
  if (blockIdx.x == 0) scan_begin_args(hdr, a, hdr_out, desc_out, reset_stats);
  classify_points<true>(hdr.total, 1u, a.d, sc);
}

// octahedral direction bin of (dx, dy, dz), 2^b x 2^b bins in Morton order
// (b = 3..6)
__device__ __forceinline__ uint32_t dir_bin(int32_t dx, int32_t dy, int32_t dz, uint32_t b) {
  const float ax = fabsf((float)dx), ay = fabsf((float)dy), az = fabsf((float)dz);
  const float s = ax + ay + az;
  if (s == 0.f) return 0;
  float u = (float)dx / s, v = (float)dy / s;
  if (dz < 0) {
    const float uu = (1.f - fabsf(v)) * (u >= 0.f ? 1.f : -1.f);
    const float vv = (1.f - fabsf(u)) * (v >= 0.f ? 1.f : -1.f);
    u = uu;
    v = vv;
  }
  const float half = (float)(1u << (b - 1u));
  const uint32_t top = (1u << b) - 1u;
  uint32_t iu = (uint32_t)((u + 1.f) * half), iv = (uint32_t)((v + 1.f) * half);
  iu = iu > top ? top : iu;
  iv = iv > top ? top : iv;
  uint32_t key = 0;
#pragma unroll
  for (int k = 0; k < 6; ++k) key |= (((iu >> k) & 1u) << (2 * k)) | (((iv >> k) & 1u) << (2 * k + 1));
  return key;
}

// Winner order of ScanScratch::ray_order: 2^b x 2^b direction bins, 2^cb
// length classes, the top hb bits of the direction (Morton) above the class
// (2b + cb = kDirBits)
struct RayOrder {
  uint32_t b, cb, hb;
};
__device__ __forceinline__ RayOrder ray_order(uint32_t k) {
  switch (k) {
    case 1: return {5u, 2u, 0u};
    case 2: return {4u, 4u, 0u};
    case 3: return {4u, 4u, 3u};
    case 4: return {4u, 4u, 4u};
    case 5: return {5u, 2u, 3u};
    default: return {6u, 0u, 0u};
  }
}

constexpr uint32_t kLeafLater = 0xFFFFFFFEu;  // tpos: the endpoint's leaf is not looked up yet

// Phase 2 (per point): the lowest-index point of each claimed voxel is its
// winner (probabilistic_map.cpp:30-54 lets only the first point of a voxel
// through the update_id test); winners are counted per bucket, and each
// keeps its place in its bucket, so that k_scan_scatter needs no atomics.
// The returning atomics of a wavefront are in flight together (one after the
// other, here and again in the scatter, took 10 + 23 us for 2,001 points, up
// to 64 round trips; now 8 + 6).
__global__ void __launch_bounds__(256) k_scan_winners(const BatchHdr* __restrict__ hdr,
                                                      const ScanDesc* __restrict__ sd,
                                                      ScanScratch sc) {
  const uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool win = false;
  uint32_t key = 0;
  if (gi < hdr->total) {
    const int4 r = sc.rec[gi];
    if ((r.w & kRecMarked) && gp(&sc.ep[sc.tpos[gi]])->first == (uint32_t)gi) {
      win = true;
      const uint32_t s = (uint32_t)r.w >> 16;
      const ScanDesc& d = sd[s];
      const uint32_t tag = s & ((1u << hdr->tag_bits) - 1u);
      const int32_t dx = r.x - d.ox, dy = r.y - d.oy, dz = r.z - d.oz;
      // The ray's length class (its cell count mx against the max range, in
      // 2^cb equal parts) sits between a coarse direction sector (hb bits)
      // and the direction inside the sector.  The rays of one wavefront then
      // end at about one distance (a batch waits for its longest ray) and,
      // ending together, cross the same leaves: short rays of one direction
      // hit near objects side by side, long ones sweep the far field.  The
      // sectors keep each region of a one-scan list (one per XCD) on one part
      // of the sphere, with a share of every length.
      // A scan with under 1/8 of its points clipped at the max range (as
      // estimated by the wavefronts that counted them), a scan of a room for
      // one, keeps the direction order: there neighbouring directions end at
      // about one distance already, and the classes would only split its
      // sweep of directions.
      const bool mixed = (uint64_t)sc.counters[kClipWords + (s & 63u)] * 128u >= (uint64_t)d.n;
      const RayOrder o = ray_order(mixed ? sc.ray_order : 0u);
      const uint32_t db = 2u * o.b - o.hb;  // direction bits below the sector
      const uint32_t mx = (uint32_t)max(abs(dx), max(abs(dy), abs(dz)));
      const uint32_t lc =
          d.reach ? min((1u << o.cb) - 1u, (uint32_t)(((uint64_t)mx << o.cb) / (d.reach + 1u))) : 0u;
      const uint32_t dir = dir_bin(dx, dy, dz, o.b);
      key = (tag << kDirBits) | ((dir >> db) << (o.cb + db)) | (lc << db) | (dir & ((1u << db) - 1u));
    }
    sc.wkey[gi] = win ? key : kNone;
  }
  // the wavefront's lanes of one bucket form a group, so that its rays stay
  // together in the bucket (groups of neighbouring lanes only: update pass of
  // 64 maps 4.28 against 3.9 ms, and 350 against 120 us here)
  uint64_t pending = __ballot(win);
  uint32_t lead = 0, rank = 0, size = 0;
  while (pending) {
    const uint32_t l = (uint32_t)__ffsll((unsigned long long)pending) - 1u;
    const bool mine = win && key == (uint32_t)__builtin_amdgcn_readlane((int)key, (int)l);
    const uint64_t same = __ballot(mine);
    if (mine) {
      lead = l;
      rank = (uint32_t)__popcll(same & lanes_below());
      size = (uint32_t)__popcll(same);
    }
    pending &= ~same;
  }
  uint32_t base = 0;
  if (win && lead == lane_id()) base = add32(&sc.hist[key], size);
  base = (uint32_t)__shfl((int)base, (int)lead);
  if (win) sc.wrank[gi] = base + rank;
}

// Phase 2 of a call of one scan of few points: the winners listed in point
// order, a wavefront's together, their endpoint-table slots released, in place
// of the buckets.  A loser that reads its voxel's slot after the release sees
// no index, which is not its own either.
__global__ void __launch_bounds__(256) k_scan_list_winners(const BatchHdr* __restrict__ hdr, ScanScratch sc) {
  const uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool win = false;
  EpSlot BXG_G* e = nullptr;
  if (gi < hdr->total && (sc.rec[gi].w & kRecMarked)) {
    e = gp(&sc.ep[sc.tpos[gi]]);
    win = e->first == (uint32_t)gi;
  }
  const uint64_t wins = __ballot(win);
  uint32_t base = 0;
  if (lane_id() == 0 && wins) base = add32(&sc.counters[0], (uint32_t)__popcll(wins));
  base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
  if (!win) return;
  sc.winners[base + (uint32_t)__popcll(wins & lanes_below())] = (uint32_t)gi;
  e->key = kEmptyKey;
  e->first = kNone;
  sc.tpos[gi] = kLeafLater;
}

// inclusive prefix sum over the 64 lanes of a wavefront
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
  const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
  for (uint32_t o = 1; o < 64u; o <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)v, o);
    if (lane >= o) v += t;
  }
  return v;
}

// Phase 2s (per bucket tile): sum of the winners of each tile of kScanTile
// buckets, four buckets a thread.
__global__ void __launch_bounds__(1024) k_scan_bucket_reduce(const BatchHdr* __restrict__ hdr,
                                                             ScanScratch sc) {
  __shared__ uint32_t wsum[16];
  const uint32_t nb = 1u << (kDirBits + hdr->tag_bits);
  const uint32_t base = blockIdx.x * kScanTile;
  if (base >= nb) return;
  const uint4 v = reinterpret_cast<const uint4*>(sc.hist + base)[threadIdx.x];
  const uint32_t s = wave_scan(v.x + v.y + v.z + v.w);
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  if (lane == 63) wsum[wid] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < 16; ++w) t += wsum[w];
    sc.counters[kTileWords + blockIdx.x] = t;
  }
}

// Calls of up to this many bucket tiles (a scan a tile) have no pass for the
// tile sums: each tile adds up the earlier ones itself (a launch saved, about
// 5 us; with more tiles the sums would take longer than the launch).
constexpr uint32_t kUnreducedTiles = 8;

// Phase 2s' (per bucket tile): exclusive scan of the bucket counts into the
// buckets' first places, carried over the earlier tiles; the last tile writes
// the winner count to counters[0].
__global__ void __launch_bounds__(1024) k_scan_bucket_scan(const BatchHdr* __restrict__ hdr,
                                                           ScanScratch sc) {
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t carry;
  const uint32_t nb = 1u << (kDirBits + hdr->tag_bits);
  const uint32_t base = blockIdx.x * kScanTile;
  if (base >= nb) return;
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  const bool reduced = gridDim.x > kUnreducedTiles;
  uint32_t sum = 0;  // this thread's part of the earlier tiles
  if (reduced) {
    // blockIdx.x < kTiles <= 64: one lane per earlier tile
    if (threadIdx.x < blockIdx.x) sum = sc.counters[kTileWords + threadIdx.x];
  } else {
    for (uint32_t t = 0; t < blockIdx.x; ++t) {
      const uint4 e = reinterpret_cast<const uint4*>(sc.hist + t * kScanTile)[threadIdx.x];
      sum += e.x + e.y + e.z + e.w;
    }
  }
  if (threadIdx.x == 0) carry = 0;
  const uint4 v = reinterpret_cast<const uint4*>(sc.hist + base)[threadIdx.x];
  const uint32_t s = v.x + v.y + v.z + v.w;
  const uint32_t incl = wave_scan(s);
  if (lane == 63) wsum[wid] = incl;
  sum = wave_scan(sum);
  __syncthreads();
  if (lane == 63 && sum) atomicAdd(&carry, sum);
  if (wid == 0) {
    const uint32_t w = lane < 16u ? wsum[lane] : 0u;
    const uint32_t wi = wave_scan(w);
    if (lane < 16u) wsum[lane] = wi;
  }
  __syncthreads();
  uint32_t run = carry + (wid ? wsum[wid - 1] : 0u) + incl - s;
  uint4 o;
  o.x = run; run += v.x;
  o.y = run; run += v.y;
  o.z = run; run += v.z;
  o.w = run;
  reinterpret_cast<uint4*>(sc.offs + base)[threadIdx.x] = o;
  if (base + kScanTile >= nb && threadIdx.x == 1023) sc.counters[0] = carry + wsum[15];
}

// Phase 2t (per point): winners written into their buckets, and their
// endpoint-table slots released (every point has read its slot by now).
// kOne: a call of one scan (one tile of buckets), whose workgroups each scan
// the 4096 bucket counts themselves, in LDS: no passes for the bucket sums.
template <bool kOne>
__global__ void __launch_bounds__(256) k_scan_scatter(const BatchHdr* __restrict__ hdr,
                                                      ScanScratch sc) {
  __shared__ uint32_t first[kOne ? kScanTile : 1];
  __shared__ uint32_t wsum[4];
  const uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t key = gi < hdr->total ? sc.wkey[gi] : kNone;
  const uint32_t rank = key != kNone ? sc.wrank[gi] : 0u;
  const uint32_t t = key != kNone ? sc.tpos[gi] : 0u;
  if (kOne) {
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    constexpr uint32_t kPer = kScanTile / 256 / 4;  // uint4s a thread
    const uint4* h = reinterpret_cast<const uint4*>(sc.hist) + threadIdx.x * kPer;
    uint4 v[kPer];
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      v[k] = h[k];
      s += v[k].x + v[k].y + v[k].z + v[k].w;
    }
    const uint32_t incl = wave_scan(s);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    uint32_t run = incl - s;
    for (uint32_t w = 0; w < wid; ++w) run += wsum[w];
    uint4* f = reinterpret_cast<uint4*>(first) + threadIdx.x * kPer;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      uint4 o;
      o.x = run; run += v[k].x;
      o.y = run; run += v[k].y;
      o.z = run; run += v[k].z;
      o.w = run; run += v[k].w;
      f[k] = o;
    }
    if (blockIdx.x == 0 && threadIdx.x == 255) sc.counters[0] = run;
    __syncthreads();
  }
  if (key == kNone) return;
  sc.winners[(kOne ? first[key] : sc.offs[key]) + rank] = (uint32_t)gi;
  EpSlot BXG_G* e = gp(&sc.ep[t]);
  e->key = kEmptyKey;
  e->first = kNone;
  sc.tpos[gi] = kLeafLater;
}

// cells a lane may run ahead of its wavefront's slowest ray when rays are
// walked whole: update pass (in a map empty at the scan's start, and in
// others) and leaf pass; the defaults of the tuning keys fresh_window,
// ray_window and leaf_window.  Measured on 64 scans: re-inserted 8 beats 4 and
// 16 (3.7 against 4.2 and 4.1 ms); leaf pass (since then 0.39) 64: 0.50, 16: 0.60, none: 0.49
// re-inserted, 0.92, 1.04, 0.98 ms into empty maps
constexpr int32_t kFreshWindow = 16;
constexpr int32_t kUpdateWindow = 8;
constexpr int32_t kLeafWindow = 64;

// The walk over the winner list.  A batch is 64 consecutive winners, rays of
// one map in neighbouring directions and (with the ray order of
// k_scan_winners) of about one length, so that they cross the same leaves
// and cache lines at about the same time; a wavefront walks one batch, one
// ray a lane, one leaf a step.  Which batch follows from the wavefront's
// number alone: no cursor, no work stealing (the grid holds a wavefront a
// batch, and the workgroups waiting for a free slot balance the load).
//
// A short list (one scan a call) has fewer batches than the GPU has wavefront
// slots, and a walk is a chain of dependent loads about 1.5 us a step: there a
// wavefront walks one segment of a batch (WalkPlan).  In a long list the rays
// are walked whole, in lockstep: a lane more than the window's cells ahead of
// the wavefront's slowest ray waits a step.
//
// Measured against persistent wavefronts that took rays from 8 cursors and
// refilled their lanes one by one in short lists (us a call; leaf pass /
// update pass): 2,001-point scan 61 / 31 -> 14 / 25, 307k-point depth frame
// 70 / 61 -> 10 / 14, 65k-point LiDAR scan at 50 m 210 / 385 -> 40 / 224;
// 64 maps 1149 / 4538 -> 500 / 3750 (leaf pass with its want bits).  Bound:
// the dependent loads of a step (entry, cells) and the scattered lines they
// touch.
//
// whether a lane at cell k steps with its wavefront: every lane that has a ray
// and is less than win cells ahead of the slowest
__device__ __forceinline__ bool in_window(bool have, int32_t k, int32_t win) {
  const bool go = have && k < wave_min(have ? k : 0x7fffffff) + win;
  return __ballot(go) == 0 ? have : go;  // else a window that wraps past 2^31
}

// the update walk of a wavefront's rays (lanes with have set); cells written
// (counted form)
template <bool kCount, class Walk>
__device__ __forceinline__ uint32_t walk_cells(const MapView& m, Walk& w, bool have, bool lockstep, int32_t win,
                                               int32_t cur, uint32_t lbase, uint32_t mark) {
  RootCache rc;
  rc.reset();
  uint32_t next_leaf = kNone, nupd = 0;
  if (have) next_leaf = walk_leaf(m, w, rc);
  while (__ballot(have)) {
    const bool go = lockstep ? in_window(have, w.k, win) : have;
    if (go) {
      nupd += apply_step<kCount>(m, w, rc, cur, lbase, mark, next_leaf);
      have = !w.done();
    }
  }
  return nupd;
}

// kMode 0: leaf allocation pass; 1: update pass; 2: counted update.
template <int kMode>
__device__ void walk_winners(const ScanDesc* __restrict__ sd, const ScanScratch& sc) {
  constexpr bool kLeaves = kMode == 0;
  const uint32_t nwin = sc.counters[0];
  const uint32_t nb = (nwin + 63u) >> 6;
  // the wavefront's number among those of its XCD (the grid is a multiple of
  // kXcds workgroups)
  const uint32_t wpb = blockDim.x >> 6;
  const uint32_t xcd = blockIdx.x % kXcds;
  const uint32_t wave = (blockIdx.x / kXcds) * wpb +
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t waves = (gridDim.x / kXcds) * wpb;
  const uint32_t lane = lane_id();
  const WalkPlan plan(nb, waves * kXcds);
  const uint32_t lg = plan.lg;
  const bool lockstep = plan.whole();
  uint32_t batch, seg;
  for (uint32_t j = wave; plan.task(j, xcd, batch, seg); j += waves) {
    if (batch >= nb) continue;
    const uint32_t idx = batch * 64u + lane;
    const bool valid = idx < nwin;
    const uint32_t gi = valid ? sc.winners[idx] : 0u;
    const int4 r = valid ? sc.rec[gi] : make_int4(0, 0, 0, 0);
    const uint32_t s = (uint32_t)r.w >> 16;
    // one scan at a time (a batch seldom holds two), so that the scan's and
    // the map's header sit in scalar registers
    uint64_t pending = __ballot(valid);
    while (pending) {
      const uint32_t s0 =
          (uint32_t)__builtin_amdgcn_readlane((int)s, __ffsll((unsigned long long)pending) - 1);
      const bool act = valid && s == s0;
      pending &= ~__ballot(act);
      const ScanDesc& d = sd[s0];
      const MapView m = uniform_view(d.map);
      const int32_t cur = uniform_i32(&m.ctr->cur);
      const uint32_t lbase = (uint32_t)uniform_i32((const int32_t*)&m.ctr->leaf_base);
      const uint32_t mark = mark_miss((uint32_t)uniform_i32((const int32_t*)&m.ctr->life));
      if (!kLeaves && (map_status(m) & kFatal)) continue;
      const int32_t win = kLeaves ? sc.win_leaves : (lbase == 0 ? sc.win_fresh : sc.win_cells);
      const int32_t ox = d.ox, oy = d.oy, oz = d.oz;
      const bool no_rays = (d.flags & kScanNoRays) != 0;
      RayWalk w;
      w.init(ox, oy, oz, r.x, r.y, r.z);
      // the update pass walks cells [0, mx) of the ray (none for an endpoint
      // in the origin's voxel or a scan without rays); the leaf pass also the
      // endpoint's cell mx, so that it creates the winner's endpoint leaf
      // (only that cell for a scan without rays)
      bool have = act && (kLeaves || !no_rays);
      const int32_t last = w.mx + (kLeaves ? 1 : 0);
      // segment seg of n = 2^lg walks cells [ceil(seg last / n), ceil((seg +
      // 1) last / n)): segment 0 holds cell 0, and they cover the ray once
      const int64_t up = (1ll << lg) - 1;
      int32_t k0 = (int32_t)(((int64_t)last * seg + up) >> lg);
      int32_t k1 = (int32_t)(((int64_t)last * (seg + 1u) + up) >> lg);
      if (no_rays) {
        k0 = w.mx;
        k1 = seg == 0 ? last : k0;
      }
      if (k0 >= k1) have = false;
      if (have) {
        if (k0 == 0)
          w.kend = k1;  // from the origin (and mx may be 0: no division)
        else
          w.seek(k0, k1);
      }
      const uint32_t ncells = have ? (uint32_t)(w.kend - w.k) : 0u;
      uint32_t nupd = 0;
      if (kLeaves) {  // walks leaves, not cells
        LeafWalk lw;
        if (have) lw.init(w, m.lb, m.ib);
        int32_t slot = kNoRoot;
        while (__ballot(have)) {
          const bool go = lockstep ? in_window(have, lw.k, win) : have;
          leaves_step(m, lw, slot, lbase == 0 ? m.want : m.have, go);
          have = have && !(go && lw.done());
        }
      } else if (__ballot(have && w.mx > kRay32)) {
        nupd = walk_cells<kMode == 2>(m, w, have, lockstep, win, cur, lbase, mark);
      } else {
        RayWalk16 w16;
        if (have) w16.init(w, m.lb);
        nupd = walk_cells<kMode == 2>(m, w16, have, lockstep, win, cur, lbase, mark);
      }
      if (kMode == 2 && ncells) {
        add64(&m.ctr->stat_ray_updates, nupd);
        add64(&m.ctr->stat_rays, seg == 0 ? 1u : 0u);
        add64(&m.ctr->stat_ray_visits, ncells);
      }
    }
  }
}

// Phase 2b: the leaves on every winner's ray that do not exist yet are put
// down as wants (k_scan_new_entries creates them before any cell is written,
// so a pool overflow leaves the map's cells untouched).
__global__ void __launch_bounds__(256) k_scan_ray_leaves(const ScanDesc* __restrict__ sd,
                                                         ScanScratch sc) {
  walk_winners<0>(sd, sc);
}

// Phase 2c (one block per scan): leaves of the rays still due from
// addHitPoint / addMissPoint calls made since the map's last insert.
__global__ void __launch_bounds__(256) k_scan_extra_leaves(const BatchHdr* __restrict__ hdr,
                                                           const ScanDesc* __restrict__ sd) {
  if (blockIdx.x >= hdr->nscans) return;
  const ScanDesc& d = sd[blockIdx.x];
  if (d.flags & kScanNoRays) return;
  const MapView m = load_view(d.map);
  // whole wavefronts: leaves_step is a wavefront collective
  for (uint32_t j0 = threadIdx.x & ~63u; j0 < d.nextra; j0 += blockDim.x) {
    const uint32_t j = j0 + lane_id();
    const int4 e = j < d.nextra ? d.extra[j] : make_int4(d.ox, d.oy, d.oz, 0);
    bool have = !(e.x == d.ox && e.y == d.oy && e.z == d.oz);
    RayWalk w;
    w.init(d.ox, d.oy, d.oz, e.x, e.y, e.z);
    LeafWalk lw;
    lw.init(w, m.lb, m.ib);
    int32_t slot = kNoRoot;
    while (__ballot(have)) {
      leaves_step(m, lw, slot, m.have, have);
      if (have && lw.done()) have = false;
    }
  }
}

// Phase 2d (per root directory word of each scan's map): the leaves wanted by
// the leaf pass are created (allocateLeafGrid and GridBlockAllocator::
// allocateBlock, bonxai.hpp:572-586 and grid_allocator.hpp:94-123): a
// wavefront takes the words of 64 inner cells that have wants, reads their
// entries, takes one bump of the map's leaf counter for up to
// kEntryRun words, writes origins and entries and the have bits, and clears
// the wants.  Entries that hold a leaf after all (have bits are hints) are
// passed over.  A map whose pool is too small is flagged, the entries past
// its end stay EMPTY, and no cell has been written (the host grows the pool
// and runs the call again).  Bound: reading the want words of the whole
// directory (8 KB a 1,024-root directory), then a chain of loads, one
// atomic and stores.
constexpr uint32_t kEntryRun = 8;
__global__ void __launch_bounds__(256) k_scan_new_entries(const BatchHdr* __restrict__ hdr,
                                                          const ScanDesc* __restrict__ sd) {
  const uint32_t lane = lane_id();
  const uint32_t wave = blockIdx.x * (blockDim.x >> 6) +
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t nwaves = gridDim.x * (blockDim.x >> 6);
  const uint32_t nscans = hdr->nscans;
  uint32_t turn = wave;  // the maps' words follow each other round the wavefronts
  for (uint32_t s = 0; s < nscans; ++s) {
    const MapView m = uniform_view(sd[s].map);
    const uint32_t ew = entry_words(m.isz);
    const uint64_t nwords = (uint64_t)(m.root_mask + 1) * ew;
    const uint32_t first = turn;
    turn = (turn + nwaves - (uint32_t)((nwords / 64) % nwaves)) % nwaves;
    for (uint64_t e0 = (uint64_t)first * 64; e0 < nwords; e0 += (uint64_t)nwaves * 64) {
      const uint64_t want = m.want[e0 + lane];  // nwords is a multiple of 64
      uint64_t pending = __ballot(want != 0);
      if (!pending) continue;
      if (want) m.want[e0 + lane] = 0;
      while (pending) {
        uint32_t l[kEntryRun], child[kEntryRun];
        uint64_t make[kEntryRun];
#pragma unroll
        for (uint32_t k = 0; k < kEntryRun; ++k) {
          l[k] = pending ? (uint32_t)__ffsll((unsigned long long)pending) - 1u : 64u;
          pending &= pending - 1;
          // a word's 64 entries (fewer in small inner grids), one a lane
          child[k] = l[k] < 64u && lane < m.isz ? m.children[(e0 + l[k]) / ew * m.isz + (e0 + l[k]) % ew * 64 + lane]
                                                : 0u;
        }
        uint32_t n = 0;
#pragma unroll
        for (uint32_t k = 0; k < kEntryRun; ++k) {
          make[k] = l[k] < 64u ? lane_value(want, l[k]) & __ballot(child[k] == kEmptyChild) : 0ull;
          n += (uint32_t)__popcll(make[k]);
        }
        uint32_t base = 0;
        if (n && lane == 0) base = add32(&m.ctr->leaf_count, n);
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
#pragma unroll
        for (uint32_t k = 0; k < kEntryRun; ++k) {
          if (l[k] >= 64u) continue;
          const uint64_t e = e0 + l[k];
          const uint32_t slot = (uint32_t)(e / ew), ci = (uint32_t)(e % ew) * 64u + lane;
          const uint32_t idx = base + (uint32_t)__popcll(make[k] & lanes_below());
          const bool mine = (make[k] >> lane) & 1ull;
          if (mine && idx < m.leaf_cap) {
            int32_t x, y, z;
            unpack_root(m.root_keys[slot], m.log2n, &x, &y, &z);
            const uint32_t im = (1u << m.ib) - 1;
            m.origin[idx] = make_int4(x + (int32_t)((ci & im) << m.lb), y + (int32_t)(((ci >> m.ib) & im) << m.lb),
                                      z + (int32_t)((ci >> (2 * m.ib)) << m.lb), (int32_t)slot);
            m.children[(uint64_t)slot * m.isz + ci] = idx;
            child[k] = idx;
          }
          const uint64_t have = __ballot(lane < m.isz && child[k] < kPendingChild);
          if (lane == 0) m.have[e] = have;
          if (mine && idx >= m.leaf_cap) or32(&m.ctr->status, kStOutOfPool);
          base += (uint32_t)__popcll(make[k]);
        }
      }
    }
  }
}

// Endpoint updates of the maps, counted by a wavefront while it stays with one
// map and added by the workgroup at the end, once a map.  (An add a wavefront
// is an atomic on one address about every 6 ns: 100k new endpoints 20 us, now
// 10; the endpoints of a LiDAR scan in old leaves 14 us, now 9.)
struct EndpointCount {
  MapCounters* map;  // the same in every lane, like the counts
  uint32_t n, back;
  __device__ __forceinline__ static void put(MapCounters* c, uint32_t n, uint32_t back) {
    if (n) add64(&c->stat_endpoint_updates, (uint64_t)n);
    if (back) add64(&c->stat_ray_updates, (uint64_t)0 - (uint64_t)back);
  }
  // every lane of the wavefront: lanes with updated set count for *ctr, and
  // those with retracted set take back a ray update
  __device__ __forceinline__ void add(bool updated, bool retracted, MapCounters* ctr) {
    uint64_t pending = __ballot(updated);
    while (pending) {
      const int leader = __ffsll((unsigned long long)pending) - 1;
      MapCounters* lc = (MapCounters*)lane_value((uint64_t)ctr, (uint32_t)leader);
      const uint64_t same = __ballot(updated && ctr == lc);
      if (lc != map) {
        if (lane_id() == 0 && map) put(map, n, back);
        map = lc;
        n = back = 0;
      }
      n += (uint32_t)__popcll(same);
      back += (uint32_t)__popcll(__ballot(retracted && ctr == lc));
      pending &= ~same;
    }
  }
  // every thread of the workgroup (at most 4 wavefronts)
  __device__ __forceinline__ void finish() {
    __shared__ EndpointCount waves[4];
    const uint32_t t = threadIdx.x, nw = blockDim.x >> 6;
    if ((t & 63u) == 0) waves[t >> 6] = *this;
    __syncthreads();
    if (t >= nw || !waves[t].map) return;
    EndpointCount c = waves[t];
    for (uint32_t w = 0; w < nw; ++w) {
      if (w == t || waves[w].map != c.map) continue;
      if (w < t) return;  // counted there
      c.n += waves[w].n;
      c.back += waves[w].back;
    }
    put(c.map, c.n, c.back);
  }
};

// Phase 3 (per winner of a map not empty at the scan's start): endpoint
// hit/miss update (probabilistic_map.cpp:30-54) of the endpoints in leaves
// that existed before the scan.  One writer per endpoint cell.  An endpoint
// in a leaf the scan created is left for k_scan_new_endpoints (after the ray
// pass): its leaf index goes to tpos.  In a map empty at the scan's start
// every endpoint leaf is new, and k_scan_new_endpoints looks it up (tpos
// stays kLeafLater): there is nothing to do here.
__global__ void __launch_bounds__(256) k_scan_endpoints(const ScanDesc* __restrict__ sd,
                                                        ScanScratch sc) {
  const uint32_t nwin = sc.counters[0];
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t start = blockIdx.x * blockDim.x + threadIdx.x;
  // every lane runs the same number of iterations so that the count below
  // sees a converged wavefront
  EndpointCount count{nullptr, 0u, 0u};
  for (uint32_t base = start - (start & 63u); base < nwin; base += stride) {
    const uint32_t idx = base + (start & 63u);
    bool updated = false;
    MapCounters* ctr = nullptr;
    if (idx < nwin) {
      const uint32_t gi = sc.winners[idx];
      const int4 r = sc.rec[gi];
      const ScanDesc& d = sd[(uint32_t)r.w >> 16];
      const MapView m = load_view(d.map);
      const uint32_t lbase = *gp(&m.ctr->leaf_base);
      const bool skip = lbase == 0 || (map_status(m) & kFatal) != 0;
      const uint32_t leaf = skip ? kNone : find_leaf(m, r.x, r.y, r.z);
      const bool fresh = leaf != kNone && leaf >= lbase;
      if (!skip) sc.tpos[gi] = fresh ? leaf : kNone;
      if (leaf != kNone && !fresh) {
        const uint32_t li = leaf_index(r.x, r.y, r.z, m.lb);
        uint32_t BXG_G* cell = (uint32_t BXG_G*)m.cells + (uint64_t)leaf * m.lsz + li;
        const uint32_t w = *cell;
        const int32_t cur = map_cur(m);
        *cell = (r.w & kRecHit) ? cell_hit(w, m.hit, m.cmax, cur) : cell_miss(w, m.miss, m.cmin, cur);
        if (w == 0) or64((uint64_t*)&m.masks[(uint64_t)leaf * m.lw + (li >> 6)], 1ull << (li & 63));
        updated = true;
        ctr = m.ctr;
      }
    }
    count.add(updated, false, ctr);
  }
  count.finish();
}

// Phase 4d (per winner): the endpoint update of the endpoints in leaves the
// scan created (k_scan_endpoints left their leaf index in tpos, or
// kLeafLater in maps empty at the scan's start).  Such a cell held zero before the scan, so its endpoint word is cell_hit(0) or
// cell_miss(0), whatever ray marked it meanwhile (the reference updates
// endpoints first and its rays skip them, probabilistic_map.cpp:30-54,
// 81-89): its touched byte becomes the hit or the miss mark, one writer per
// voxel, and k_scan_new_leaves writes the word.  The counted form takes back
// the ray update the ray pass counted for a cell that turns out to be an
// endpoint.
// It also zeroes the bucket counts for the next call.
template <bool kCount>
__global__ void __launch_bounds__(256) k_scan_new_endpoints(const BatchHdr* __restrict__ hdr,
                                                            const ScanDesc* __restrict__ sd,
                                                            ScanScratch sc) {
  const uint32_t nwin = sc.counters[0];
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t start = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nb4 = (1u << (kDirBits + hdr->tag_bits)) / 4;
  for (uint32_t i = start; i < nb4; i += stride)
    reinterpret_cast<uint4*>(sc.hist)[i] = make_uint4(0u, 0u, 0u, 0u);
  EndpointCount count{nullptr, 0u, 0u};
  for (uint32_t base = start - (start & 63u); base < nwin; base += stride) {
    const uint32_t idx = base + (start & 63u);
    bool updated = false, retracted = false;
    MapCounters* ctr = nullptr;
    if (idx < nwin) {
      const uint32_t gi = sc.winners[idx];
      uint32_t leaf = sc.tpos[gi];
      const int4 r = sc.rec[gi];
      const MapView m = load_view(sd[(uint32_t)r.w >> 16].map);
      if (leaf == kLeafLater) leaf = (map_status(m) & kFatal) ? kNone : find_leaf(m, r.x, r.y, r.z);
      if (leaf != kNone) {
        uint8_t BXG_G* tb = m.touched + (uint64_t)leaf * m.lsz + leaf_index(r.x, r.y, r.z, m.lb);
        const uint32_t life = *gp(&m.ctr->life);
        if (kCount) retracted = *tb == mark_miss(life);
        *tb = (uint8_t)((r.w & kRecHit) ? mark_hit(life) : mark_miss(life));
        updated = true;
        ctr = m.ctr;
      }
    }
    count.add(updated, retracted, ctr);
  }
  count.finish();
}

// Phase 4: the ray clear of updateFreeCells (probabilistic_map.cpp:77-101):
// every cell of Ray(origin, endpoint) takes the miss update unless its
// update_id already equals the scan's id.
template <bool kCount>
__global__ void __launch_bounds__(256) k_scan_rays(const ScanDesc* __restrict__ sd,
                                                   ScanScratch sc) {
  walk_winners<kCount ? 2 : 1>(sd, sc);
}

// Phase 4b (one block per scan): rays due from addHitPoint / addMissPoint.
template <bool kCount>
__global__ void __launch_bounds__(256) k_scan_extra_rays(const BatchHdr* __restrict__ hdr,
                                                         const ScanDesc* __restrict__ sd) {
  if (blockIdx.x >= hdr->nscans) return;
  const ScanDesc& d = sd[blockIdx.x];
  if (d.flags & kScanNoRays) return;
  const MapView m = load_view(d.map);
  if (map_status(m) & kFatal) return;
  const int32_t cur = map_cur(m);
  const uint32_t lbase = *gp(&m.ctr->leaf_base);
  const uint32_t mark = mark_miss(*gp(&m.ctr->life));
  for (uint32_t j = threadIdx.x; j < d.nextra; j += blockDim.x) {
    const int4 e = d.extra[j];
    if (e.x == d.ox && e.y == d.oy && e.z == d.oz) continue;
    RayWalk w;
    RootCache rc;
    rc.reset();
    w.init(d.ox, d.oy, d.oz, e.x, e.y, e.z);
    uint32_t n = 0;
    uint32_t next_leaf = walk_leaf(m, w, rc);
    while (!w.done()) n += apply_step<kCount>(m, w, rc, cur, lbase, mark, next_leaf);
    if (kCount) {
      add64(&m.ctr->stat_ray_updates, n);
      add64(&m.ctr->stat_rays, 1);
      add64(&m.ctr->stat_ray_visits, (uint32_t)w.mx);
    }
  }
}

// Phase 4c: the leaves the scan created, written whole.  Their cells were
// all off before the scan (a created leaf is initialised, as the reference's
// Grid constructor does, bonxai.hpp:51-58), and the scan left in each
// cell's touched byte what it did there: the life's miss mark (a ray, or a
// miss endpoint: cell_miss(0)), its hit mark (a hit endpoint: cell_hit(0)), or
// neither (nothing).  So every cell word follows from its byte, and the mask
// is exactly the marked bytes (Accessor::value(create) sets the bit,
// bonxai.hpp:485-490): one pass per new leaf writes its cells and mask words,
// with no read of the cell pool and no atomic.  (Clearing the marks here took
// 2.78 ms for a frame's 4.12M new leaves; marks that belong to a life need no
// clearing: 2.43 ms, 4.5 TB/s of the 10.8 GB.)  The new leaves of each scan's
// map are [leaf_base, leaf_count); those of a failed call are written off
// (zero).  Bound: HBM.
//
// Phase 5 (per scan) on the first workgroup, whose results no other
// workgroup of this kernel reads: update_count 1 -> 2 -> 3 -> 1
// (probabilistic_map.cpp:103-105) unless the scan failed; every scanned map's
// counters to its pinned host mirror, so that the host learns pool use and
// errors from one event after the call (no copy a map); the winner count and
// the clip counts back to zero.
__device__ __forceinline__ void scan_finalize(uint32_t nscans, const ScanDesc* sd, const ScanScratch& sc) {
  if (threadIdx.x < 64u) sc.counters[kClipWords + threadIdx.x] = 0;
  if (threadIdx.x == 0) sc.counters[0] = 0;
  for (uint32_t s = threadIdx.x; s < nscans; s += blockDim.x) {
    const MapDev BXG_G* md = (const MapDev BXG_G*)sd[s].map;
    MapCounters BXG_G* ctr = gp(md->ctr);
    if (!(sd[s].flags & kScanNoRays) && !(ctr->status & kFatal)) {
      const int32_t c = ctr->cur + 1;
      ctr->cur = c == 4 ? 1 : c;
      ctr->scans_applied += 1;
    }
    const uint64_t BXG_G* src = (const uint64_t BXG_G*)ctr;
    uint64_t* dst = (uint64_t*)md->ctr_host;
    uint64_t v[sizeof(MapCounters) / 8];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(MapCounters) / 8; ++k) v[k] = src[k];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(MapCounters) / 8; ++k) dst[k] = v[k];
  }
}

constexpr uint32_t kNewLeafRun = 4;  // leaves a wavefront of k_scan_new_leaves has in flight
__global__ void __launch_bounds__(256) k_scan_new_leaves(const BatchHdr* __restrict__ hdr,
                                                         const ScanDesc* __restrict__ sd, ScanScratch sc) {
  if (blockIdx.x == 0) scan_finalize(hdr->nscans, sd, sc);
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
  const uint32_t nscans = hdr->nscans;
  for (uint32_t s = 0; s < nscans; ++s) {
    const MapView m = load_view(sd[s].map);
    const MapCounters BXG_G* ctr = gp(m.ctr);
    const uint32_t lo = ctr->leaf_base;
    const uint32_t hi = min(ctr->leaf_count, m.leaf_cap);
    if (lo >= hi) continue;
    const int32_t cur = ctr->scan_cur;
    // a failed call's leaves stay off: no byte is its mark
    const bool failed = (ctr->status & kFatal) != 0;
    const uint32_t bmiss = failed ? ~0u : mark_miss(ctr->life);
    const uint32_t bhit = failed ? ~0u : mark_hit(ctr->life);
    const uint32_t wmiss = cell_miss(0u, m.miss, m.cmin, cur);
    const uint32_t whit = cell_hit(0u, m.hit, m.cmax, cur);
    if (m.lsz == 512) {
      // 8^3 leaves (the default leaf_bits 3): lane l has cells 4l..4l+3 and
      // 256+4l..256+4l+3, so each store instruction writes 1 KB in one piece
      // (measured: 2.98 ms a fresh frame's new leaves, against 3.63 ms with
      // 8 consecutive cells a lane).  The cell stores are nontemporal: a
      // frame's new leaves (8.4 GB) would only push its other data out of
      // the caches (2.52 ms against 2.98 ms).
      for (uint32_t leaf0 = lo + wave; leaf0 < hi; leaf0 += kNewLeafRun * nwaves) {
        uint32_t t[kNewLeafRun][2];
#pragma unroll
        for (uint32_t k = 0; k < kNewLeafRun; ++k) {
          const uint32_t leaf = leaf0 + k * nwaves;
          const uint32_t BXG_G* tp = (const uint32_t BXG_G*)(m.touched + (uint64_t)leaf * 512u) + lane;
          t[k][0] = leaf < hi ? tp[0] : 0u;  // (0 is no life's mark)
          t[k][1] = leaf < hi ? tp[64] : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < kNewLeafRun; ++k) {
          const uint32_t leaf = leaf0 + k * nwaves;
          if (leaf >= hi) break;  // uniform across the wavefront
#pragma unroll
          for (uint32_t h = 0; h < 2; ++h) {
            uint32_t v[4];
            uint32_t nib = 0;
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
              const uint32_t cls = (t[k][h] >> (8 * b)) & 0xFFu;
              v[b] = cls == bmiss ? wmiss : (cls == bhit ? whit : 0u);
              nib |= ((cls == bmiss) | (cls == bhit) ? 1u : 0u) << b;
            }
            u32x4 BXG_G* cp = (u32x4 BXG_G*)(m.cells + (uint64_t)leaf * 2048u + 1024u * h) + lane;
            __builtin_nontemporal_store(u32x4{v[0], v[1], v[2], v[3]}, cp);
            // mask word 4h + r: the nibbles of lanes 16r..16r+15, lane 16r + i
            // at bits 4i..4i+3; lanes 16r..16r+7 fill the low half, 16r+8..
            // 16r+15 the high half.  OR over each half-row of 8 lanes (DPP
            // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror), then lane 16r
            // takes the high half from lane 16r+8 (row_ror:8).
            const uint32_t sh = 4u * (lane & 7u);
            uint32_t mlo = (lane & 8u) ? 0u : nib << sh;
            uint32_t mhi = (lane & 8u) ? nib << sh : 0u;
            mlo |= (uint32_t)__builtin_amdgcn_update_dpp((int)mlo, (int)mlo, 0xB1, 0xF, 0xF, false);
            mhi |= (uint32_t)__builtin_amdgcn_update_dpp((int)mhi, (int)mhi, 0xB1, 0xF, 0xF, false);
            mlo |= (uint32_t)__builtin_amdgcn_update_dpp((int)mlo, (int)mlo, 0x4E, 0xF, 0xF, false);
            mhi |= (uint32_t)__builtin_amdgcn_update_dpp((int)mhi, (int)mhi, 0x4E, 0xF, 0xF, false);
            mlo |= (uint32_t)__builtin_amdgcn_update_dpp((int)mlo, (int)mlo, 0x141, 0xF, 0xF, false);
            mhi |= (uint32_t)__builtin_amdgcn_update_dpp((int)mhi, (int)mhi, 0x141, 0xF, 0xF, false);
            mhi = (uint32_t)__builtin_amdgcn_update_dpp((int)mhi, (int)mhi, 0x128, 0xF, 0xF, false);
            if ((lane & 15u) == 0u)
              m.masks[(uint64_t)leaf * 8u + 4u * h + (lane >> 4)] = ((uint64_t)mhi << 32) | mlo;
          }
        }
      }
    } else {
      for (uint32_t leaf = lo + wave; leaf < hi; leaf += nwaves) {
        const uint8_t BXG_G* tb = m.touched + (uint64_t)leaf * m.lsz;
        uint32_t BXG_G* cells = (uint32_t BXG_G*)m.cells + (uint64_t)leaf * m.lsz;
        for (uint32_t w = 0; w < m.lw; ++w) {
          const uint32_t i = w * 64u + lane;
          const uint32_t cls = i < m.lsz ? tb[i] : 0u;
          if (i < m.lsz) cells[i] = cls == bmiss ? wmiss : (cls == bhit ? whit : 0u);
          const uint64_t b = __ballot((cls == bmiss) | (cls == bhit));
          if (lane == 0) m.masks[(uint64_t)leaf * m.lw + w] = b;
        }
      }
    }
  }
}

// After a scan that ran out of nodes (it wrote no cell): the overflow bits
// are cleared and the bump counter, which ran past the pool, comes back to
// the pool's size.  The leaves allocated below it stay, every cell off.
__global__ void k_na_recover(MapCounters* __restrict__ ctr, uint32_t leaf_cap) {
  if (threadIdx.x != 0) return;
  ctr->status &= ~(kStOutOfPool | kStRootFull);
  ctr->leaf_count = min(ctr->leaf_count, leaf_cap);
}

// ------------------------------------------------------ bulk cell ops

// setValue / setCellOn / setCellOff for a batch, with the results of the calls
// made one after the other (bonxai.hpp:449-466, 537-569).  Two kernels:
// k_op_tiles orders each tile of inputs by the bucket (hash) of their leaf (of
// 512 cells of it in leaves of 16^3, op_unit_log), and k_op_buckets gives each
// bucket to one workgroup, which finds the first and last input of every cell in
// LDS.  Such a unit belongs to one workgroup, so its cells and (of up to
// kOpGathered units a bucket) its mask words need no device atomics, and the
// workgroup initialises the leaves it creates.
//
// A table of the cells in device memory (claim, last index, mask bits: two to
// three device atomics an input, about 15 G/s in all) took 0.46 ms for 2M
// inputs into a new grid, clear and leaf initialisation included, and five
// launches; the two kernels take 0.030 + 0.058 ms (0.4 MB of bucket starts
// aside, 64 bytes an input are moved: 1.4 TB/s).  What bounds them: the tiles'
// claims of missing roots (12 us) and their passes through LDS; in the
// buckets a chain of some ten dependent reads a workgroup with two or three
// workgroups a CU (reads of the entries 14 us, LDS tables 6, leaves looked up
// and created 13, values and cells 17).

constexpr uint32_t kOpTileThreads = 1024;
constexpr uint32_t kOpTileLog = 13;    // most inputs of a tile
constexpr uint32_t kOpMaxBuckets = 4096;
constexpr uint32_t kOpThreads = 512;   // of k_op_buckets (2M inputs: 256 threads 93 us, 512 66, 1024 102)
// Most units of a bucket whose mask bits are gathered in LDS: clusters of cells
// have some 54 a bucket.  With more, few cells share a word: 1M inputs, each in a
// leaf of its own, 977 a bucket, are set in 122 us, call and wait included, with
// an atomic a cell, and in 448 when buckets were done in parts of at most 256
// leaves.
constexpr uint32_t kOpGathered = 256;

enum : uint32_t { kOpSetValue = 0, kOpSetOn = 1, kOpSetOff = 2 };

struct OpScratch {
  uint64_t* entry;   // per tile, its inputs by bucket: cell << kOpTileLog | place in the tile
  uint16_t* start;   // per tile, each bucket's first entry, nb + 1 words (stride nb + 2)
  uint32_t tile;     // inputs a tile
  uint32_t tiles;
  uint32_t nb;       // buckets (a power of two, 8 or more)
};

// a key of an LDS table: the slot's key, or kEmptyKey taken by this key
__device__ __forceinline__ uint64_t lds_claim(uint64_t* p, uint64_t key) {
  uint64_t k = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (k != kEmptyKey) return k;
  k = atomicCAS((unsigned long long*)p, kEmptyKey, key);
  return k == kEmptyKey ? key : k;
}
__device__ __forceinline__ uint32_t lds_claim(uint32_t* p, uint32_t key) {
  uint32_t k = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (k != kNone) return k;
  k = atomicCAS(p, kNone, key);
  return k == kNone ? key : k;
}

// The inputs of a tile in the order of their leaves' buckets.  kCreate:
// missing roots are created (setCellOff leaves out inputs without one), and the
// map's leaf count before the call is kept (k_op_buckets).  The tile's distinct
// roots are found in LDS and looked up once.
//
// A tile in which one bucket has an eighth of the inputs or more leaves out
// those of it that no result needs.  Else the one workgroup of that bucket reads
// them all, one after the other: 2M inputs in one leaf 2.76 ms, now 0.096 (in one
// cell 2.75, now 0.061); 2M, half of them in one leaf, 1.45, now 0.15; 50k in one
// leaf 105 us, now 42.
template <bool kCreate, int kPer>
__global__ void __launch_bounds__(kOpTileThreads) k_op_tiles(const MapDev* __restrict__ mp,
                                                             const int32_t* __restrict__ coords, uint64_t n,
                                                             uint32_t op, uint8_t* __restrict__ was_on,
                                                             OpScratch os) {
  constexpr uint32_t kTile = kOpTileThreads * kPer;
  constexpr uint32_t kRoots = kTile * 2 < 4096 ? kTile * 2 : 4096;
  constexpr uint32_t kStage = kTile * 8 > kRoots * 12 ? kTile * 8 : kRoots * 12;
  constexpr uint32_t kCrowd = kTile / 8;  // inputs of a bucket that is looked at for inputs to leave out
  constexpr uint32_t kDups = kStage >= 65536 ? 4096 : kStage >= 32768 ? 2048 : 1024;  // their table
  static_assert(kDups * 16 <= kStage, "the table of cells");
  __shared__ __attribute__((aligned(16))) uint8_t stage[kStage];
  __shared__ uint32_t hist[kOpMaxBuckets / 2];  // 16 bits a bucket
  __shared__ uint32_t wsum[kOpTileThreads / 64];
  __shared__ uint32_t crowded;
  uint64_t* rkeys = (uint64_t*)stage;
  int32_t* rslots = (int32_t*)(stage + kRoots * 8);
  const MapView m = uniform_view(mp);
  const uint32_t t = threadIdx.x, lane = t & 63u, wid = t >> 6;
  const uint64_t base = (uint64_t)blockIdx.x * kTile;
  const bool count = kCreate && blockIdx.x == 0 && t == 0;
  const uint32_t leaves = count ? min(*gp(&m.ctr->leaf_count), m.leaf_cap) : 0u;
  for (uint32_t p = t; p < kRoots; p += kOpTileThreads) rkeys[p] = kEmptyKey;
  for (uint32_t p = t; p < os.nb / 2; p += kOpTileThreads) hist[p] = 0;
  if (t == 0) crowded = 0;
  int32_t x[kPer], y[kPer], z[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint64_t i = base + (uint32_t)j * kOpTileThreads + t;
    x[j] = y[j] = z[j] = 0;
    if (i < n) {
      const int32_t BXG_G* c = gp(coords) + 3 * i;
      x[j] = c[0];
      y[j] = c[1];
      z[j] = c[2];
      if (was_on) was_on[i] = op == kOpSetOff ? 0 : 1;
    }
  }
  __syncthreads();
  if (count) m.ctr->leaf_base = leaves;
  constexpr uint32_t kOut = 0xFFFFFFFFu, kDirect = 0xFFFFFFFEu;
  uint32_t rp[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    rp[j] = kOut;
    if (base + (uint32_t)j * kOpTileThreads + t < n) {
      uint64_t key;
      if (!pack_root(x[j], y[j], z[j], m.log2n, &key)) {
        if (kCreate) or32(&m.ctr->status, kStCoordRange);
      } else {
        uint32_t h = (uint32_t)mix64(key) & (kRoots - 1);
        rp[j] = kDirect;  // a table with no room near: the input asks the map itself
        for (int p = 0; p < 16; ++p) {
          if (lds_claim(&rkeys[h], key) == key) {
            rp[j] = h;
            break;
          }
          h = (h + 1) & (kRoots - 1);
        }
      }
    }
  }
  __syncthreads();
  // Workgroups begin at different parts of their tables: those that start
  // together then claim different roots of a new grid, and find the rest
  // claimed (2M cells in 1,584 new roots: 42 -> 30 us)
  for (uint32_t q = t; q < kRoots; q += kOpTileThreads) {
    const uint32_t p = (q + blockIdx.x * kOpTileThreads) & (kRoots - 1u);
    const uint64_t key = rkeys[p];
    bool inserted = false;
    if (key != kEmptyKey) rslots[p] = kCreate ? root_probe(m, key, inserted) : root_find(m, key);
    const uint64_t b = __ballot(inserted);
    if (b && lane == 0) add32(&m.ctr->root_count, (uint32_t)__popcll(b));
  }
  __syncthreads();
  const uint32_t cl = 3 * m.lb, il = 3 * m.ib, ul = op_unit_log(m.lb);
  uint64_t ent[kPer];
  uint32_t at[kPer];  // bucket << 16 | rank in the tile's part of it
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    int32_t slot = -1;
    if (rp[j] < kRoots) {
      slot = rslots[rp[j]];
    } else if (rp[j] == kDirect) {
      uint64_t key;
      pack_root(x[j], y[j], z[j], m.log2n, &key);
      bool inserted = false;
      slot = kCreate ? root_probe(m, key, inserted) : root_find(m, key);
      if (inserted) add32(&m.ctr->root_count, 1u);
    }
    at[j] = kOut;
    if (slot >= 0) {
      const uint64_t child = ((uint64_t)slot << il) | inner_index(x[j], y[j], z[j], m.lb, m.ib);
      const uint64_t cell = (child << cl) | leaf_index(x[j], y[j], z[j], m.lb);
      const uint32_t bk = (uint32_t)mix64(cell >> ul) & (os.nb - 1);
      const uint32_t sh = (bk & 1u) * 16u;
      const uint32_t r = atomicAdd(&hist[bk >> 1], 1u << sh) >> sh & 0xFFFFu;
      if (r + 1u == kCrowd) crowded = 1;
      ent[j] = (cell << kOpTileLog) | ((uint32_t)j * kOpTileThreads + t);
      at[j] = (bk << 16) | r;
    }
  }
  __syncthreads();
  if (crowded) {
    // Only the first (was_on is asked for, or setCellOn / setCellOff) and the
    // last input (setValue) of a cell have a part in the results.  Cells that
    // find no room in the table keep all their inputs.
    uint64_t* cells = (uint64_t*)stage;
    uint32_t* first = (uint32_t*)(stage + kDups * 8);
    uint32_t* last = first + kDups;
    for (uint32_t p = t; p < kDups; p += kOpTileThreads) {
      cells[p] = kEmptyKey;
      first[p] = kNone;
      last[p] = 0;
    }
    __syncthreads();
    const bool need_last = op == kOpSetValue, need_first = !need_last || was_on != nullptr;
    uint32_t dup[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      dup[j] = kOut;
      if (at[j] == kOut) continue;
      const uint32_t bk = at[j] >> 16;
      if (((hist[bk >> 1] >> ((bk & 1u) * 16u)) & 0xFFFFu) < kCrowd) continue;
      const uint64_t cell = ent[j] >> kOpTileLog;
      uint32_t h = op_cell_slot(cell) & (kDups - 1u);
      for (int p = 0; p < 16; ++p) {
        if (lds_claim(&cells[h], cell) == cell) {
          dup[j] = h;
          atomicMin(&first[h], (uint32_t)j * kOpTileThreads + t);
          atomicMax(&last[h], (uint32_t)j * kOpTileThreads + t);
          break;
        }
        h = (h + 1u) & (kDups - 1u);
      }
    }
    __syncthreads();
    for (uint32_t p = t; p < os.nb / 2; p += kOpTileThreads) hist[p] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (at[j] == kOut) continue;
      const uint32_t bk = at[j] >> 16, sh = (bk & 1u) * 16u, here = (uint32_t)j * kOpTileThreads + t;
      at[j] = kOut;
      if (dup[j] != kOut && !(need_last && last[dup[j]] == here) && !(need_first && first[dup[j]] == here)) continue;
      at[j] = (bk << 16) | (atomicAdd(&hist[bk >> 1], 1u << sh) >> sh & 0xFFFFu);
    }
    __syncthreads();
  }
  // first places of the buckets: two words (four buckets) a thread
  constexpr uint32_t kMost = kOpMaxBuckets / 2 / kOpTileThreads;
  const uint32_t nw = os.nb / 2;
  uint32_t c[kMost], sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < kMost; ++k) {
    const uint32_t w = t * kMost + k;
    c[k] = w < nw ? hist[w] : 0u;
    sum += (c[k] & 0xFFFFu) + (c[k] >> 16);
  }
  const uint32_t incl = wave_scan(sum);
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  uint32_t run = incl - sum;
  for (uint32_t w = 0; w < wid; ++w) run += wsum[w];
  uint32_t* start = (uint32_t*)(os.start + (uint64_t)blockIdx.x * (os.nb + 2));
#pragma unroll
  for (uint32_t k = 0; k < kMost; ++k) {
    const uint32_t w = t * kMost + k;
    if (w < nw) {
      const uint32_t lo = run, hi = run + (c[k] & 0xFFFFu);
      run = hi + (c[k] >> 16);
      hist[w] = lo | (hi << 16);
      start[w] = lo | (hi << 16);
      if (w == nw - 1) start[nw] = run;  // the tile's inputs in all
    }
  }
  __syncthreads();
  uint64_t* sorted = (uint64_t*)stage;
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if (at[j] != kOut) {
      const uint32_t bk = at[j] >> 16;
      sorted[((hist[bk >> 1] >> ((bk & 1u) * 16u)) & 0xFFFFu) + (at[j] & 0xFFFFu)] = ent[j];
    }
  __syncthreads();
  uint32_t total = 0;
  for (uint32_t w = 0; w < kOpTileThreads / 64; ++w) total += wsum[w];
  for (uint32_t p = t; p < total; p += kOpTileThreads) gp(os.entry)[base + p] = sorted[p];
}

// A value of vb bytes, or zero bytes: in the widest words that the caller's
// buffer (at `at`: every value lies at a multiple of vb from it) and the size
// allow, several on their way together.  (A byte at a time, 500k lookups of
// 64-byte cells, one a thread, took 830 us, now 38; as many set 353, now 58.)
template <class W, uint32_t kTogether>
__device__ __forceinline__ void copy_words(uint8_t BXG_G* dst, const uint8_t BXG_G* src, uint32_t n, bool on) {
  W BXG_G* d = (W BXG_G*)dst;
  const W BXG_G* s = (const W BXG_G*)src;
  uint32_t k = 0;
  for (; k + kTogether <= n; k += kTogether) {
    W v[kTogether] = {};
    if (on) {
#pragma unroll
      for (uint32_t j = 0; j < kTogether; ++j) v[j] = s[k + j];
    }
#pragma unroll
    for (uint32_t j = 0; j < kTogether; ++j) d[k + j] = v[j];
  }
  for (; k < n; ++k) d[k] = on ? s[k] : W{};
}
__device__ __forceinline__ void copy_value(uint8_t BXG_G* dst, const uint8_t BXG_G* src, uint32_t vb,
                                           const void* at, bool on = true) {
  const uint32_t odd = (uint32_t)(uintptr_t)at | vb;
  if ((odd & 15u) == 0)
    copy_words<u32x4, 4>(dst, src, vb / 16, on);
  else if ((odd & 3u) == 0)
    copy_words<uint32_t, 4>(dst, src, vb / 4, on);
  else
    copy_words<uint8_t, 4>(dst, src, vb, on);
}

// whether values of vb bytes at vals can be read as words
__device__ __forceinline__ bool whole_words(const uint8_t* vals, uint32_t vb) {
  return (vb == 4 || vb == 8) && ((uintptr_t)vals & (vb - 1u)) == 0;
}

// A bucket of a bulk call.  kCreate: its missing leaves are created, all cells
// off and zero (bonxai.hpp:51-58).  kApply: its cells are set.  Without kApply
// (the pass before, for calls that the pool may be too small for) nothing is
// done where the pool has room for a leaf an input after all.  kFirst: the
// call needs each cell's first input and prior mask bit (was_on is asked for,
// or setCellOn / setCellOff); a setValue batch without was_on needs only the
// last input of each cell.  was_on of an input is the prior bit for the first
// of its cell and "on" (off for setCellOff) for later ones, which k_op_tiles
// has written; setValue keeps the last input's value, setCellOn the first
// one's, if the cell was off.
//
// A bucket with more cells or units than the tables hold is done in parts
// (OpPart).  The table of the units has room for the inputs of a bucket that
// lie each in a leaf of its own.  Up to kOpGathered units are numbered, have a
// thread each, and their cells' mask bits are gathered in LDS and written by
// one thread a word; the bits of more units by an atomic a cell (they share
// few words then).  Leaves of several units are created without kApply only,
// each by the workgroup that claims it.
template <bool kCreate, bool kApply, bool kFirst, bool kLast>
__global__ void __launch_bounds__(kOpThreads, kFirst && kLast ? 4 : 6) k_op_buckets(const MapDev* __restrict__ mp,
                                                           const uint8_t* __restrict__ vals, uint64_t n,
                                                           uint32_t op, uint8_t* __restrict__ was_on,
                                                           OpScratch os) {
  constexpr uint32_t kCells = kApply ? kOpCells : 4;
  // cells: the unit's slot << kOpUnitLog | cell in the unit
  __shared__ __attribute__((aligned(16))) uint32_t ckey[kCells];
  __shared__ __attribute__((aligned(16))) uint32_t clast[kLast ? kOpCells : 4];
  __shared__ __attribute__((aligned(16))) uint32_t cfirst[kFirst ? kOpCells : 4];
  // the units (entry among the children, place in the leaf), then what became of them (below)
  __shared__ __attribute__((aligned(16))) uint64_t leaf[kOpLeaves];
  // of the numbered units: unit and slot, then what became of them
  __shared__ uint64_t gathered[kApply ? kOpGathered : 1];
  // the mask words of the numbered units, in place of inputs that are read by then
  uint64_t* bits = (uint64_t*)(kLast ? clast : cfirst);
  static_assert(kOpCells * 4 >= kOpGathered * 8 << (kOpUnitLog - 6u), "their mask words");
  __shared__ uint32_t leaves_full, cells_full, nleaf, nnew, nbase, fatal;
  const MapView m = uniform_view(mp);
  const uint32_t t = threadIdx.x, lane = t & 63u, wid = t >> 6;
  const uint32_t il = 3 * m.ib, ul = op_unit_log(m.lb), sl = 3 * m.lb - ul;  // 2^sl units a leaf
  if (kCreate && !kApply && sl == 0 && (uint64_t)*gp(&m.ctr->leaf_base) + n <= m.leaf_cap) return;
  // A failed call sets no cell.  The status is read once for the workgroup (and
  // looked at behind the first barriers): its wavefronts go through the same
  // ones whatever other workgroups flag.
  if (t == 0) fatal = map_status(m) & kFatal;
  // buckets that follow each other (their entries share lines) on one XCD
  const uint32_t bk = (blockIdx.x % kXcds) * (os.nb / kXcds) + blockIdx.x / kXcds;
  const uint32_t lwl = ul > 6u ? ul - 6u : 0u;  // log2 of a unit's mask words
  // lanes a tile, so that the workgroup reads all tiles' entries at once (more
  // than 64 in calls of few tiles: 2,000 inputs in one leaf 40 us with 64, now 28)
  uint32_t gl = 0;
  while (((uint64_t)os.tiles << gl) < kOpThreads) ++gl;
  constexpr uint32_t kMine = kOpCells / kOpThreads, kMyLeaves = kOpLeaves / kOpThreads;
  // what became of a unit: its leaf's index (kNone: there is none), its number <<
  // 32 (below kOpGathered), its place in the leaf << kPartBit, kMade if this
  // kernel has created the leaf
  constexpr uint64_t kMade = 1ull << 63;
  constexpr uint32_t kPartBit = 40;
  static_assert(kOpGathered <= 256, "a unit's number");
  const auto part_of = [](uint64_t w) -> uint32_t { return (uint32_t)(w >> kPartBit) & 7u; };
  constexpr uint32_t kSlotBit = 48;  // a unit is below 2^39
  constexpr uint32_t kTogether = 4;
  const auto table = [](const auto* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const auto cell_key = [&](uint64_t cell, uint32_t ls) -> uint32_t {
    return (ls << kOpUnitLog) | ((uint32_t)cell & ((1u << ul) - 1u));
  };
  // a leaf's or cell's slot, from the first on that may hold it; false if none
  // of kOpProbes does
  const auto claim_leaf = [&](uint64_t unit, uint32_t& ls) -> bool {
    for (uint32_t p = 0; p < kOpProbes; ++p) {
      uint64_t k = __hip_atomic_load(&leaf[ls], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (k == kEmptyKey) {
        k = atomicCAS((unsigned long long*)&leaf[ls], kEmptyKey, unit);
        if (k == kEmptyKey) {
          k = unit;
          const uint32_t number = atomicAdd(&nleaf, 1u);
          if (kApply && number < kOpGathered) gathered[number] = unit | ((uint64_t)ls << kSlotBit);
        }
      }
      if (k == unit) return true;
      ls = (ls + 1u) & (kOpLeaves - 1u);
    }
    return false;
  };
  const auto claim_cell = [&](uint32_t key, uint32_t& h) -> bool {
    for (uint32_t p = 0; p < kOpProbes; ++p) {
      if (lds_claim(&ckey[h], key) == key) return true;
      h = (h + 1u) & (kOpCells - 1u);
    }
    return false;
  };
  OpPart part;
  for (;;) {
    const uint4 ones = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (kApply) {
      for (uint32_t p = t; p < kOpCells / 4; p += kOpThreads) {
        reinterpret_cast<uint4*>(ckey)[p] = ones;  // kNone
        if (kLast) reinterpret_cast<uint4*>(clast)[p] = make_uint4(0u, 0u, 0u, 0u);
        if (kFirst) reinterpret_cast<uint4*>(cfirst)[p] = ones;
      }
    }
    for (uint32_t p = t; p < kOpLeaves / 2; p += kOpThreads) reinterpret_cast<uint4*>(leaf)[p] = ones;  // kEmptyKey
    if (t == 0) leaves_full = cells_full = nleaf = nnew = 0;
    __syncthreads();
    const bool whole = part.whole();
    for (uint32_t tile = t >> gl; tile < os.tiles; tile += kOpThreads >> gl) {
      const uint16_t BXG_G* st = gp((const uint16_t*)os.start) + (uint64_t)tile * (os.nb + 2) + bk;
      const uint32_t hi = st[1];
      const uint64_t tb = (uint64_t)tile * os.tile;
      const uint64_t BXG_G* entry = gp((const uint64_t*)os.entry) + tb;
      const auto input = [&](uint64_t e) -> uint32_t { return (uint32_t)tb + ((uint32_t)e & ((1u << kOpTileLog) - 1u)); };
      const bool crowd = whole && hi - st[0] >= (8u << gl);
      for (uint32_t k = st[0] + (t & ((1u << gl) - 1u)); k < hi;) {
        uint32_t n_here = 1, todo = 1;  // inputs k, k + (1 << gl), ...; bits of those not in the tables yet
        if (crowd && k + ((kTogether - 1u) << gl) < hi) {
          // of a leaf that takes a large part of the call's inputs, all of them
          // this workgroup's, most are: kTogether at a time, so that as many
          // chains of reads are under way
          uint64_t e[kTogether];
          bool known[kTogether];
#pragma unroll
          for (uint32_t j = 0; j < kTogether; ++j) e[j] = entry[k + (j << gl)];
#pragma unroll
          for (uint32_t j = 0; j < kTogether; ++j) {
            const uint64_t unit = e[j] >> (kOpTileLog + ul);
            known[j] = table(&leaf[op_leaf_slot(unit)]) == unit;
          }
          if (kApply) {
#pragma unroll
            for (uint32_t j = 0; j < kTogether; ++j) {
              const uint64_t cell = e[j] >> kOpTileLog;
              known[j] &= table(&ckey[op_cell_slot(cell)]) == cell_key(cell, op_leaf_slot(cell >> ul));
            }
          }
          n_here = kTogether;
          todo = 0;
#pragma unroll
          for (uint32_t j = 0; j < kTogether; ++j) {
            if (!known[j]) {
              todo |= 1u << j;
            } else if (kApply) {
              const uint32_t h = op_cell_slot(e[j] >> kOpTileLog);
              if (kLast) atomicMax(&clast[h], input(e[j]));
              if (kFirst) atomicMin(&cfirst[h], input(e[j]));
            }
          }
        }
        for (; todo; todo &= todo - 1u) {
          const uint64_t e = entry[k + (((uint32_t)__ffs((int)todo) - 1u) << gl)], cell = e >> kOpTileLog, unit = cell >> ul;
          if (!whole && !part.holds(mix64(unit), mix64(cell))) continue;
          uint32_t ls = op_leaf_slot(unit);
          if (!claim_leaf(unit, ls)) {
            leaves_full = 1;
            continue;
          }
          if (!kApply) continue;
          uint32_t h = op_cell_slot(cell);
          if (!claim_cell(cell_key(cell, ls), h)) {
            cells_full = 1;
            continue;
          }
          if (kLast) atomicMax(&clast[h], input(e));
          if (kFirst) atomicMin(&cfirst[h], input(e));
        }
        k += n_here << gl;
      }
    }
    __syncthreads();
    if (leaves_full | cells_full) {
      const bool more = part.halve(leaves_full != 0);
      __syncthreads();
      if (more) continue;
      if (t == 0) or32(&m.ctr->status, kStScratchFull);  // cells of one hash: not met
      return;
    }
    const bool failed = fatal != 0;
    if (kApply && failed && was_on)
      for (uint64_t i = (uint64_t)blockIdx.x * kOpThreads + t; i < n; i += (uint64_t)gridDim.x * kOpThreads)
        was_on[i] = 0;
    if (!kCreate && failed) return;
    // the values of the cells, in flight while the leaves are looked up (or the
    // inputs that hold them), and the words of `bits` cleared
    const bool word = whole_words(vals, m.vb);
    uint32_t* inputs = kLast ? clast : cfirst;
    std::conditional_t<kLast, uint64_t, uint32_t> val[kMine] = {};
    if (kApply && !failed) {
      uint32_t src[kMine];  // (empty slots: input 0)
#pragma unroll
      for (uint32_t j = 0; j < kMine; ++j) src[j] = inputs[j * kOpThreads + t];
#pragma unroll
      for (uint32_t j = 0; j < kMine; ++j) inputs[j * kOpThreads + t] = 0;
      if (kLast && word && m.vb == 4) {
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) val[j] = gp((const uint32_t*)vals)[src[j]];
      } else if (kLast && word) {
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) val[j] = gp((const uint64_t*)vals)[src[j]];
      } else {
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) val[j] = src[j];
      }
    }
    // the leaves: looked up, and created where missing
    const uint32_t nl = nleaf;
    const bool gather = kApply && nl <= kOpGathered;
    // the thread's j-th unit
    const auto unit_of = [&](uint32_t j) -> uint64_t {
      if (!gather) return leaf[j * kOpThreads + t];
      return j == 0 && t < nl ? gathered[t] & ((1ull << kSlotBit) - 1ull) : kEmptyKey;
    };
    uint32_t idx[kMyLeaves];
    uint32_t have = 0, make = 0, at = 0;  // its leaves and those missing (bits), the first new one's place
#pragma unroll
    for (uint32_t j = 0; j < kMyLeaves; ++j) {
      const uint64_t unit = unit_of(j);
      have |= unit != kEmptyKey ? 1u << j : 0u;
      idx[j] = unit != kEmptyKey ? m.children[unit >> sl] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < kMyLeaves; ++j) {
      if (idx[j] < kPendingChild) continue;
      // a leaf of several units belongs to the workgroup that claims it
      if (!kApply && sl && !leaf_claim((uint32_t*)&m.children[unit_of(j) >> sl], idx[j])) continue;
      make |= 1u << j;
    }
    if (kCreate) {
      if (make) at = atomicAdd(&nnew, (uint32_t)__popc(make));
      __syncthreads();
      const uint32_t k = nnew;
      if (k) {
        if (t == 0) nbase = add32(&m.ctr->leaf_count, k);
        __syncthreads();
        const uint32_t first = nbase;
        uint32_t next = first + at;
#pragma unroll
        for (uint32_t j = 0; j < kMyLeaves; ++j) {
          if (!((make >> j) & 1u)) continue;
          const uint64_t child = unit_of(j) >> sl;
          idx[j] = next++;
          if (idx[j] >= m.leaf_cap) {
            or32(&m.ctr->status, kStOutOfPool);
            idx[j] = kNone;
            st32((uint32_t*)&m.children[child], kEmptyChild);
            continue;
          }
          const uint32_t ci = (uint32_t)child & (m.isz - 1u), im = (1u << m.ib) - 1u;
          int32_t ox, oy, oz;
          unpack_root(m.root_keys[child >> il], m.log2n, &ox, &oy, &oz);
          m.origin[idx[j]] =
              make_int4(ox + (int32_t)((ci & im) << m.lb), oy + (int32_t)(((ci >> m.ib) & im) << m.lb),
                        oz + (int32_t)((ci >> (2 * m.ib)) << m.lb), (int32_t)(child >> il));
          st32((uint32_t*)&m.children[child], idx[j]);
        }
        const bool masks = !gather || failed;  // else written below
        const uint32_t cw = (uint32_t)((uint64_t)m.lsz * m.vb / 8);  // 8-byte words a leaf
        for (uint32_t r = first + wid; r < first + k && r < m.leaf_cap; r += kOpThreads / 64) {
          if (masks)
            for (uint32_t w = lane; w < m.lw; w += 64) m.masks[(uint64_t)r * m.lw + w] = 0;
          for (uint32_t w = lane; w < cw; w += 64) ((uint64_t BXG_G*)m.cells)[(uint64_t)r * cw + w] = 0;
        }
      }
    }
    if (kApply && !failed) {
#pragma unroll
      for (uint32_t j = 0; j < kMyLeaves; ++j) {
        if (!((have >> j) & 1u)) continue;
        uint64_t w = idx[j] < kPendingChild ? idx[j] : kNone;
        if (kCreate && ((make >> j) & 1u)) w |= kMade;
        w |= (unit_of(j) & ((1ull << sl) - 1ull)) << kPartBit;
        if (gather) {
          leaf[gathered[t] >> kSlotBit] = w | ((uint64_t)t << 32);
          gathered[t] = w;
        } else {
          leaf[j * kOpThreads + t] = w;
        }
      }
      __syncthreads();
      // the prior mask bits, read together
      uint32_t pres = 0;
      if (kFirst) {
        uint64_t masks[kMine];
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) {
          const uint32_t key = ckey[j * kOpThreads + t];
          const uint64_t l = key != kNone ? leaf[key >> kOpUnitLog] : (uint64_t)kNone;
          masks[j] = 0;
          if ((uint32_t)l != kNone && !(kCreate && (l & kMade)))
            masks[j] = m.masks[(uint64_t)(uint32_t)l * m.lw + (part_of(l) << lwl) + ((key & ((1u << kOpUnitLog) - 1u)) >> 6)];
        }
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) pres |= (uint32_t)(masks[j] >> (ckey[j * kOpThreads + t] & 63u) & 1u) << j;
      }
#pragma unroll
      for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t p = j * kOpThreads + t, key = ckey[p], lu = key & ((1u << kOpUnitLog) - 1u);
        if (key == kNone) continue;
        const uint64_t l = leaf[key >> kOpUnitLog];
        const uint32_t at_leaf = (uint32_t)l;
        if (at_leaf == kNone) continue;
        const uint32_t li = part_of(l) << ul | lu;
        const uint64_t g = (uint64_t)at_leaf * m.lsz + li;
        const uint64_t bit = 1ull << (li & 63u);
        uint64_t* mw = (uint64_t*)&m.masks[(uint64_t)at_leaf * m.lw + (li >> 6)];
        const bool pre = kFirst && ((pres >> j) & 1u);
        if (kFirst && was_on) was_on[kLast ? cfirst[p] : (uint32_t)val[j]] = pre;
        if (word && (kLast || op == kOpSetOff || (vals && !pre))) {
          uint64_t v = kLast ? (uint64_t)val[j] : 0ull;
          if (!kLast && vals) v = m.vb == 4 ? gp((const uint32_t*)vals)[val[j]] : gp((const uint64_t*)vals)[val[j]];
          if (m.vb == 4)
            ((uint32_t BXG_G*)m.cells)[g] = (uint32_t)v;
          else
            ((uint64_t BXG_G*)m.cells)[g] = v;
        }
        if (gather) {
          atomicOr((unsigned long long*)&bits[((uint32_t)(l >> 32 & 0xFFu) << lwl) + (lu >> 6)], bit);
        } else if (op == kOpSetOff) {
          if (pre) and64(mw, ~bit);
        } else if (!pre) {
          or64(mw, bit);
        }
      }
      __syncthreads();
      if (gather) {
        for (uint32_t w = t; w < (nl << lwl); w += kOpThreads) {
          const uint64_t v = bits[w], l = gathered[w >> lwl];
          if ((uint32_t)l == kNone) continue;
          uint64_t BXG_G* mw = m.masks + (uint64_t)(uint32_t)l * m.lw + (part_of(l) << lwl) + (w & ((1u << lwl) - 1u));
          if (kCreate && (l & kMade))
            *mw = v;  // every word of a new leaf
          else if (v)
            *mw = op == kOpSetOff ? *mw & ~v : *mw | v;
        }
      }
      // cells of other sizes, and values at any address (inputs: own slots again)
      if (m.vb && !word && (op != kOpSetOn || vals)) {
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j)
          inputs[j * kOpThreads + t] = op == kOpSetOn && ((pres >> j) & 1u) ? kNone : (uint32_t)val[j];
#pragma unroll 1
        for (uint32_t p = t; p < kOpCells; p += kOpThreads) {
          const uint32_t key = ckey[p], src = inputs[p];
          const uint64_t l = key != kNone && src != kNone ? leaf[key >> kOpUnitLog] : (uint64_t)kNone;
          if ((uint32_t)l == kNone) continue;
          const uint64_t g = (uint64_t)(uint32_t)l * m.lsz + (part_of(l) << ul | (key & ((1u << kOpUnitLog) - 1u)));
          copy_value(m.cells + g * m.vb, gp(vals) + (uint64_t)src * m.vb, m.vb, vals, op != kOpSetOff);
        }
      }
    }
    if (!part.next()) return;
    __syncthreads();
  }
}

// create the root and leaf of every coordinate (setValue / setCellOn path)
__global__ void __launch_bounds__(256) k_touch(const MapDev* __restrict__ mp,
                                               const int32_t* __restrict__ coords, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const MapView m = load_view(mp);
  const int32_t x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
  uint64_t key;
  if (!pack_root(x, y, z, m.log2n, &key)) {
    or32(&m.ctr->status, kStCoordRange);
    return;
  }
  const int32_t slot = root_insert(m, key);
  if (slot < 0) return;
  const int32_t lmask = ~((1 << m.lb) - 1);
  leaf_request(m, (uint32_t)slot, inner_index(x, y, z, m.lb, m.ib), x & lmask, y & lmask, z & lmask);
}


// ConstAccessor::value / isCellOn (bonxai.hpp:496-534) for a batch, one
// lookup a thread: root key -> inner entry -> cell (-> mask word).  4- and
// 8-byte cells: the cell first.  Off cells hold zero bytes, so a nonzero cell
// is on and its mask word is not read; only a zero cell (off, or on with a
// zero value) costs the mask load.  Bound: the chain of loads in small
// batches, the scattered cell lines in large ones (8M random reads of a 2M-
// cell grid: 0.107 ms; the hits' 4-byte reads alone take 0.075).  Four
// lookups a thread, their loads issued together, leave too few wavefronts to
// cover the chain: 0.113 ms, 16k lookups 9 against 6 us, 64 batches of 256k
// 710 against 490 us; the mask loaded beside the cell: 0.132 ms.
__global__ void __launch_bounds__(256) k_lookup(const MapDev* __restrict__ mp,
                                                const int32_t* __restrict__ coords, uint64_t n,
                                                uint8_t* __restrict__ vals,
                                                uint8_t* __restrict__ found) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const MapView m = uniform_view(mp);
  const int32_t BXG_G* cg = gp(coords);
  const int32_t x = cg[3 * i], y = cg[3 * i + 1], z = cg[3 * i + 2];
  const uint32_t leaf = find_leaf(m, x, y, z);
  const uint32_t vb = m.vb;
  const bool cell_first = vb == 4 || vb == 8;
  uint64_t v = 0, g = 0;
  bool on = false;
  if (leaf != kNone) {
    const uint32_t li = leaf_index(x, y, z, m.lb);
    g = (uint64_t)leaf * m.lsz + li;
    if (cell_first)
      v = vb == 4 ? (uint64_t)((const uint32_t BXG_G*)m.cells)[g] : ((const uint64_t BXG_G*)m.cells)[g];
    on = v != 0 || ((m.masks[(uint64_t)leaf * m.lw + (li >> 6)] >> (li & 63)) & 1ull);
  }
  if (found) found[i] = on;
  if (!vals || !vb) return;
  if (vb == 4) {
    ((uint32_t*)vals)[i] = (uint32_t)v;
  } else if (vb == 8) {
    ((uint64_t*)vals)[i] = v;
  } else {
    copy_value(gp(vals) + i * vb, m.cells + g * vb, vb, vals, on);
  }
}

// isOccupied / isUnknown / isFree (probabilistic_map.cpp:56-75) for a batch:
// 1 occupied, -1 free, 0 unknown
__global__ void __launch_bounds__(256) k_classify_cells(const MapDev* __restrict__ mp,
                                                        const int32_t* __restrict__ coords,
                                                        uint64_t n, int8_t* __restrict__ state) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const MapView m = load_view(mp);
  const int32_t x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
  const uint32_t leaf = find_leaf(m, x, y, z);
  int8_t st = 0;
  if (leaf != kNone) {
    const uint32_t li = leaf_index(x, y, z, m.lb);
    if ((m.masks[(uint64_t)leaf * m.lw + (li >> 6)] >> (li & 63)) & 1) {
      const int32_t p = cell_p(((const uint32_t BXG_G*)m.cells)[(uint64_t)leaf * m.lsz + li]);
      st = p > m.thr ? 1 : (p < m.thr ? -1 : 0);
    }
  }
  state[i] = st;
}

// ------------------------------------------------------ whole-map passes

// forEachCell (bonxai.hpp:704-743) as a compaction; filter 0 all, 1 p >
// threshold, 2 p < threshold.  A wavefront takes `words` mask words (64 cells
// each; 4 to 32): one lane holds each word, reduced by the filter to the
// cells that pass; their popcounts place the cells, with one atomic on the
// output counter per workgroup (one per 64 cells, all on one word, took 2.39
// ms for a LiDAR map of 6.5M cells, about 6 ns an atomic; this
// form 0.07 ms, 1.9 TB/s of lists and cells).  Few words a wavefront keep
// small maps wide (a room of 2k leaves: 32 words 17 us, 4 words 7 us), many keep the
// atomics few in large ones (1024 threads of 8 words 0.16 ms, of 16 words
// 0.12 ms).  Bound: the chain of mask, count, atomic and cells in each
// workgroup, then the lists' bytes.
constexpr uint32_t kExportMostWords = 32;
constexpr uint32_t kExportBlock = 512;
constexpr uint32_t kExportRun = 4;  // words with loads in flight together
__global__ void __launch_bounds__(kExportBlock) k_export(const MapDev* __restrict__ mp, uint32_t nleaves,
                                                         uint32_t words_a_wave, uint32_t filter,
                                                         int32_t* __restrict__ coords,
                                                         uint8_t* __restrict__ vals, uint64_t cap,
                                                         uint64_t* __restrict__ count) {
  __shared__ uint32_t wbase[kExportBlock / 64];  // cells of the workgroup's earlier wavefronts
  __shared__ uint64_t base;
  __shared__ uint16_t list[kExportBlock / 64][kExportMostWords * 64];
  const MapView m = uniform_view(mp);
  const uint32_t lane = lane_id();
  const uint32_t wib = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint64_t nwords = (uint64_t)nleaves * m.lw;
  const uint64_t w0 = ((uint64_t)blockIdx.x * (kExportBlock / 64) + wib) * words_a_wave;
  const uint32_t lwl = m.lb >= 2 ? 3u * m.lb - 6u : 0u;  // log2 of the words a leaf
  uint64_t mine = lane < words_a_wave && w0 + lane < nwords ? m.masks[w0 + lane] : 0;
  if (m.lsz < 64) mine &= (1ull << m.lsz) - 1;
  const uint32_t BXG_G* words = (const uint32_t BXG_G*)m.cells;  // of 4-byte cells
  const auto cell_of = [&](uint32_t w) {  // first cell of word w0 + w
    return ((w0 + w) >> lwl) * m.lsz + (((w0 + w) & (m.lw - 1)) << 6);
  };
  if (filter) {
    for (uint32_t g = 0; g < words_a_wave; g += kExportRun) {
      uint64_t word[kExportRun];
      uint32_t v[kExportRun];
#pragma unroll
      for (uint32_t k = 0; k < kExportRun; ++k) {
        word[k] = lane_value(mine, g + k);
        v[k] = (word[k] >> lane) & 1 ? words[cell_of(g + k) + lane] : 0u;
      }
#pragma unroll
      for (uint32_t k = 0; k < kExportRun; ++k) {
        const int32_t p = cell_p(v[k]);
        const uint64_t b = __ballot(((word[k] >> lane) & 1) && (filter == 1 ? p > m.thr : p < m.thr));
        if (lane == g + k) mine = b;
      }
    }
  }
  const uint32_t c = (uint32_t)__popcll(mine);
  const uint32_t incl = wave_scan(c);
  const uint32_t before = incl - c;  // cells of the wavefront's earlier words
  if (lane == 63) wbase[wib] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < kExportBlock / 64; ++w) {
      const uint32_t n = wbase[w];
      wbase[w] = t;
      t += n;
    }
    base = t ? add64(count, t) : 0;
  }
  __syncthreads();
  const uint64_t first = base + wbase[wib];
  const uint32_t vb = vals ? m.vb : 0u;
  if (first >= cap || (!coords && !vb)) return;
  // the wavefront's cells (word, bit) listed in LDS, so that 64 of them are
  // read and written at a time however few a word holds
  for (uint32_t w = 0; w < words_a_wave; ++w) {
    const uint64_t word = lane_value(mine, w);
    if ((word >> lane) & 1)
      list[wib][(uint32_t)__builtin_amdgcn_readlane((int)before, (int)w) +
                (uint32_t)__popcll(word & lanes_below())] = (uint16_t)(w * 64u + lane);
  }
  const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
  const bool by_word = vb == 4 && ((uint64_t)vals & 3) == 0;  // caller's buffer may be unaligned
  const uint32_t lb = m.lb, lm = (1u << lb) - 1;
#pragma unroll kExportRun
  for (uint32_t i = lane; i < n; i += 64) {
    const uint64_t pos = first + i;
    if (pos >= cap) break;
    const uint32_t e = list[wib][i];
    const uint64_t word = w0 + (e >> 6);
    const uint64_t leaf = word >> lwl;
    const uint32_t li = (uint32_t)((word & (m.lw - 1)) << 6) + (e & 63u);
    const uint64_t cell = leaf * m.lsz + li;
    if (by_word)
      ((uint32_t*)vals)[pos] = words[cell];
    else if (vb)
      copy_value(gp(vals) + pos * vb, m.cells + cell * vb, vb, vals);
    if (coords) {
      const int4 o = m.origin[leaf];
      coords[3 * pos] = o.x | (int32_t)(li & lm);
      coords[3 * pos + 1] = o.y | (int32_t)((li >> lb) & lm);
      coords[3 * pos + 2] = o.z | (int32_t)((li >> (2 * lb)) & lm);
    }
  }
}

// order-free digest of the on cells (count, sum, xor, sum of remix)
__global__ void __launch_bounds__(256) k_digest(const MapDev* __restrict__ mp, uint32_t nleaves,
                                                uint64_t* __restrict__ out) {
  const MapView m = load_view(mp);
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t leaf = t >> (3 * m.lb);
  const uint32_t li = (uint32_t)(t & (m.lsz - 1));
  uint64_t h = 0, h2 = 0, c = 0;
  if (leaf < nleaves && ((m.masks[leaf * m.lw + (li >> 6)] >> (li & 63)) & 1)) {
    const int4 o = m.origin[leaf];
    const uint32_t lb = m.lb, lm = (1u << lb) - 1, vb = m.vb;
    uint64_t word = 0;
    const uint8_t BXG_G* src = m.cells + (leaf * m.lsz + li) * vb;
    if (vb <= 8) {
      for (uint32_t b = 0; b < vb; ++b) word |= (uint64_t)src[b] << (8 * b);
    } else {
      for (uint32_t off = 0; off < vb; off += 8) {
        uint64_t part = 0;
        for (uint32_t b = 0; b < 8 && off + b < vb; ++b) part |= (uint64_t)src[off + b] << (8 * b);
        word = mix64(word ^ part);
      }
    }
    h = cell_hash(o.x | (int32_t)(li & lm), o.y | (int32_t)((li >> lb) & lm),
                  o.z | (int32_t)((li >> (2 * lb)) & lm), word);
    h2 = mix64(h ^ 0xA0761D6478BD642Full);
    c = 1;
  }
  // wavefront reduction, then one atomic per wavefront
  uint64_t x = h;
  for (int off = 32; off > 0; off >>= 1) {
    c += __shfl_xor(c, off);
    h += __shfl_xor(h, off);
    x ^= __shfl_xor(x, off);
    h2 += __shfl_xor(h2, off);
  }
  if (lane_id() == 0 && c) {
    add64(&out[0], c);
    add64(&out[1], h);
    xor64(&out[2], x);
    add64(&out[3], h2);
  }
}

// activeCellsCount (bonxai.hpp:689-701): popcount of every leaf mask word
__global__ void __launch_bounds__(256) k_count_on(const MapDev* __restrict__ mp, uint32_t nleaves,
                                                  uint64_t* __restrict__ out) {
  const MapView m = load_view(mp);
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t c = 0;
  if (t < (uint64_t)nleaves * m.lw) {
    const uint64_t w = m.masks[t];
    c = m.lsz < 64 ? (uint64_t)__popcll(w & ((1ull << m.lsz) - 1)) : (uint64_t)__popcll(w);
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if (lane_id() == 0 && c) add64(out, c);
}

// clear(SET_ALL_CELLS_OFF): every mask word and every cell byte to zero
__global__ void __launch_bounds__(256) k_cells_off(const MapDev* __restrict__ mp, uint32_t nleaves) {
  const MapView m = load_view(mp);
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nw = (uint64_t)nleaves * m.lw;
  for (uint64_t w = t; w < nw; w += (uint64_t)gridDim.x * blockDim.x) m.masks[w] = 0;
  const uint64_t nb = (uint64_t)nleaves * m.lsz * m.vb / 4;
  for (uint64_t b = t; b < nb; b += (uint64_t)gridDim.x * blockDim.x) ((uint32_t BXG_G*)m.cells)[b] = 0;
}

// re-insert every root of an old directory into the (empty) directory of m;
// with prune set, roots without any leaf are dropped
__global__ void __launch_bounds__(256) k_rehash(const MapDev* __restrict__ mp,
                                                const uint64_t* __restrict__ old_keys,
                                                const uint32_t* __restrict__ old_children,
                                                uint32_t old_cap, uint32_t prune) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= old_cap) return;
  const uint64_t key = old_keys[s];
  if (key == kEmptyKey) return;
  const MapView m = load_view(mp);
  if (prune) {
    bool any = false;
    for (uint32_t c = 0; c < m.isz && !any; ++c)
      any = old_children[(uint64_t)s * m.isz + c] < kPendingChild;
    if (!any) return;
  }
  const int32_t ns = root_insert(m, key);
  if (ns < 0) return;
  for (uint32_t c = 0; c < m.isz; ++c) {
    const uint32_t leaf = old_children[(uint64_t)s * m.isz + c];
    m.children[(uint64_t)ns * m.isz + c] = leaf;
    if (leaf < kPendingChild) m.origin[leaf].w = ns;
  }
}

// ------------------------------------------ releaseUnusedMemory compaction

// live[k] = 1 if leaf k has any cell on (bonxai.hpp:367-387 keeps exactly those)
__global__ void __launch_bounds__(256) k_leaf_live(const MapDev* __restrict__ mp, uint32_t nleaves,
                                                   uint32_t* __restrict__ live) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nleaves) return;
  const MapView m = load_view(mp);
  uint64_t any = 0;
  for (uint32_t w = 0; w < m.lw; ++w) any |= m.masks[(uint64_t)k * m.lw + w];
  live[k] = any != 0;
}

// Exclusive prefix sum of n 32-bit values in tiles of kScanTile: per-tile
// sums, then a one-block scan of the tile sums, then each tile with its carry.
__global__ void __launch_bounds__(1024) k_tile_reduce(const uint32_t* __restrict__ in, uint64_t n,
                                                      uint32_t* __restrict__ tiles) {
  __shared__ uint32_t wsum[16];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + 4ull * threadIdx.x;
  uint32_t s = 0;
  for (uint32_t j = 0; j < 4; ++j) s += base + j < n ? in[base + j] : 0u;
  s = wave_scan(s);
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  if (lane == 63) wsum[wid] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < 16; ++w) t += wsum[w];
    tiles[blockIdx.x] = t;
  }
}

__global__ void __launch_bounds__(1024) k_tile_sums_scan(uint32_t* __restrict__ tiles,
                                                         uint32_t ntiles, uint32_t* __restrict__ total) {
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t carry;
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (uint32_t b = 0; b < ntiles; b += 1024) {
    const uint32_t i = b + threadIdx.x;
    const uint32_t v = i < ntiles ? tiles[i] : 0u;
    const uint32_t incl = wave_scan(v);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    if (wid == 0) {
      const uint32_t w = lane < 16u ? wsum[lane] : 0u;
      const uint32_t wi = wave_scan(w);
      if (lane < 16u) wsum[lane] = wi;
    }
    __syncthreads();
    const uint32_t excl = carry + (wid ? wsum[wid - 1] : 0u) + incl - v;
    if (i < ntiles) tiles[i] = excl;
    __syncthreads();
    if (threadIdx.x == 0) carry += wsum[15];
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}

__global__ void __launch_bounds__(1024) k_tile_scan(const uint32_t* __restrict__ in, uint64_t n,
                                                    const uint32_t* __restrict__ tiles,
                                                    uint32_t* __restrict__ out) {
  __shared__ uint32_t wsum[16];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + 4ull * threadIdx.x;
  uint32_t v[4], s = 0;
  for (uint32_t j = 0; j < 4; ++j) {
    v[j] = base + j < n ? in[base + j] : 0u;
    s += v[j];
  }
  const uint32_t incl = wave_scan(s);
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  if (wid == 0) {
    const uint32_t w = lane < 16u ? wsum[lane] : 0u;
    const uint32_t wi = wave_scan(w);
    if (lane < 16u) wsum[lane] = wi;
  }
  __syncthreads();
  uint32_t run = tiles[blockIdx.x] + (wid ? wsum[wid - 1] : 0u) + incl - s;
  for (uint32_t j = 0; j < 4; ++j) {
    if (base + j < n) out[base + j] = run;
    run += v[j];
  }
}

// Move every live leaf k to index newidx[k] of the new pool arrays and point
// its inner-grid entry there; the entries of dead leaves become empty.
// One block per old leaf.
__global__ void __launch_bounds__(256) k_compact_leaves(
    const MapDev* __restrict__ mp, uint32_t nleaves, const uint32_t* __restrict__ live,
    const uint32_t* __restrict__ newidx, uint64_t* __restrict__ dmasks, uint8_t* __restrict__ dcells,
    int4* __restrict__ dorigin) {
  const uint32_t k = blockIdx.x;
  if (k >= nleaves) return;
  const MapView m = load_view(mp);
  const int4 o = m.origin[k];
  const bool on = live[k] != 0;
  const uint32_t nk = newidx[k];
  if (threadIdx.x == 0) {
    const uint32_t ii = inner_index(o.x, o.y, o.z, m.lb, m.ib);
    m.children[(uint64_t)o.w * m.isz + ii] = on ? nk : kEmptyChild;
    if (on) dorigin[nk] = o;
  }
  if (!on) return;
  for (uint32_t w = threadIdx.x; w < m.lw; w += blockDim.x)
    dmasks[(uint64_t)nk * m.lw + w] = m.masks[(uint64_t)k * m.lw + w];
  const uint64_t nb = (uint64_t)m.lsz * m.vb;
  if (nb % 4 == 0) {
    const uint32_t BXG_G* src = (const uint32_t BXG_G*)(m.cells + (uint64_t)k * nb);
    uint32_t* dst = (uint32_t*)(dcells + (uint64_t)nk * nb);
    for (uint64_t b = threadIdx.x; b < nb / 4; b += blockDim.x) dst[b] = src[b];
  } else {
    for (uint64_t b = threadIdx.x; b < nb; b += blockDim.x)
      dcells[(uint64_t)nk * nb + b] = m.cells[(uint64_t)k * nb + b];
  }
}

// clear(CLEAR_MEMORY): directory keys and entries to all ones (kEmptyKey,
// kEmptyChild), have bits, bump counters and status to zero, the next life.  cap
// is a power of two >= 1024, so both arrays are whole 16-byte words.  Bound: HBM.
// In large directories a workgroup writes one part of each array: with all of
// them going through it side by side 2^24 roots (4.4 GB) took 1.03 ms, now 0.80,
// 2^20 46.4 us, now 44.7; 2^18 take 14.4 either way, 2^17 9.4 side by side, 10.0
// in parts.
constexpr uint64_t kClearParts = 1ull << 18;  // largest directory cleared side by side
__global__ void __launch_bounds__(256) k_map_clear(uint64_t* __restrict__ keys, uint32_t* __restrict__ children,
                                                   uint64_t* __restrict__ have, uint64_t cap, uint32_t isz,
                                                   MapCounters* __restrict__ ctr, uint32_t life) {
  static_assert(kEmptyKey == ~0ull && kEmptyChild == ~0u, "all ones");
  const uint4 ones = make_uint4(~0u, ~0u, ~0u, ~0u);
  const bool parts = cap > kClearParts;
  const auto fill = [parts](auto* p, uint64_t n, auto v) {
    const uint64_t part = parts ? (n + gridDim.x - 1) / gridDim.x : blockDim.x;
    const uint64_t end = parts ? min(n, (blockIdx.x + 1) * part) : n, step = parts ? blockDim.x : (uint64_t)gridDim.x * part;
    for (uint64_t i = blockIdx.x * part + threadIdx.x; i < end; i += step) p[i] = v;
  };
  fill(reinterpret_cast<uint4*>(keys), cap / 2, ones);
  fill(reinterpret_cast<uint4*>(children), cap * isz / 4, ones);
  if (have) fill(have, cap * entry_words(isz), (uint64_t)0);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctr->leaf_count = ctr->root_count = ctr->status = 0;
    ctr->life = life;
  }
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}
__global__ void k_fill_u64(uint64_t* p, uint64_t n, uint64_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ----------------------------------------------------- leaf page I/O

// Copy whole leaves (mask words + cell bytes) named by their origin coords
// into flat buffers; exists[k] = 0 where the leaf is absent (zeros copied).
__global__ void __launch_bounds__(256) k_read_leaves(const MapDev* __restrict__ mp,
                                                     const int32_t* __restrict__ origins, uint32_t n,
                                                     uint64_t* __restrict__ masks,
                                                     uint8_t* __restrict__ cells,
                                                     uint8_t* __restrict__ exists) {
  const MapView m = load_view(mp);
  const uint32_t k = blockIdx.x;
  if (k >= n) return;
  const uint32_t leaf = find_leaf(m, origins[3 * k], origins[3 * k + 1], origins[3 * k + 2]);
  if (threadIdx.x == 0) exists[k] = leaf != kNone;
  for (uint32_t w = threadIdx.x; w < m.lw; w += blockDim.x)
    masks[(uint64_t)k * m.lw + w] = leaf != kNone ? m.masks[(uint64_t)leaf * m.lw + w] : 0;
  const uint64_t nb = (uint64_t)m.lsz * m.vb;
  for (uint64_t b = threadIdx.x; b < nb; b += blockDim.x)
    cells[k * nb + b] = leaf != kNone ? m.cells[leaf * nb + b] : 0;
}

// Overwrite whole leaves (they must exist: run k_touch on the origins first).
// Cells whose bit is off are written as zero bytes (the off-cell invariant).
__global__ void __launch_bounds__(256) k_write_leaves(const MapDev* __restrict__ mp,
                                                      const int32_t* __restrict__ origins,
                                                      uint32_t n, const uint64_t* __restrict__ masks,
                                                      const uint8_t* __restrict__ cells) {
  const MapView m = load_view(mp);
  const uint32_t k = blockIdx.x;
  if (k >= n) return;
  const uint32_t leaf = find_leaf(m, origins[3 * k], origins[3 * k + 1], origins[3 * k + 2]);
  if (leaf == kNone) return;
  for (uint32_t w = threadIdx.x; w < m.lw; w += blockDim.x)
    m.masks[(uint64_t)leaf * m.lw + w] = masks[(uint64_t)k * m.lw + w];
  const uint32_t vb = m.vb;
  const uint64_t nb = (uint64_t)m.lsz * vb;
  for (uint64_t b = threadIdx.x; b < nb; b += blockDim.x) {
    const uint32_t li = (uint32_t)(b / vb);
    const bool on = (masks[(uint64_t)k * m.lw + (li >> 6)] >> (li & 63)) & 1;
    m.cells[leaf * nb + b] = on ? cells[k * nb + b] : 0;
  }
}

// origins of all allocated leaves (for paging a whole map to the host)
__global__ void __launch_bounds__(256) k_leaf_origins(const MapDev* __restrict__ mp, uint32_t nleaves,
                                                      int32_t* __restrict__ out) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nleaves) return;
  const MapView m = load_view(mp);
  const int4 o = m.origin[k];
  out[3 * k] = o.x;
  out[3 * k + 1] = o.y;
  out[3 * k + 2] = o.z;
}

}  // namespace bxg

// bxg_walk.h -- the integer 3-D ray walk of RayIterator
// (probabilistic_map.hpp:162-203) as the scan kernels run it, one run of
// cells inside one leaf at a time.  Plain C++ with no HIP dependence, so the
// same code compiles for the GPU (bxg_kernels.hip) and for the host check
// of tests/test_ray_walk.py.
#pragma once

#include <stdint.h>

#if defined(__HIP__)
#define BXG_HD __host__ __device__ __forceinline__
#else
#define BXG_HD inline
#endif

namespace bxg {

constexpr int kRun = 8;  // cells of one leaf handled per step of a ray
// longest ray (cells) whose closed forms fit 32 bits: a 32-bit division costs
// about a fifth of a 64-bit one
constexpr int32_t kRay32 = 32767;

// Cell 0 is the origin voxel, then max|d|-1 further cells; the end voxel is
// not part of the ray and a zero-length ray is empty.  (cx, cy, cz) is cell
// k.  The error terms are kept biased by h = ceil(mx / 2): the reference's
// "2 e >= mx" is "e - h >= 0".
struct RayWalk {
  int32_t cx, cy, cz;
  int32_t sx, sy, sz;
  int32_t dx, dy, dz;
  int32_t ex, ey, ez;  // error terms minus h
  int32_t mx, k, kend;
  BXG_HD void init(int32_t ox, int32_t oy, int32_t oz, int32_t tx, int32_t ty, int32_t tz) {
    cx = ox;
    cy = oy;
    cz = oz;
    dx = tx - ox;
    dy = ty - oy;
    dz = tz - oz;
    sx = dx < 0 ? -1 : 1;
    sy = dy < 0 ? -1 : 1;
    sz = dz < 0 ? -1 : 1;
    dx = dx < 0 ? -dx : dx;
    dy = dy < 0 ? -dy : dy;
    dz = dz < 0 ? -dz : dz;
    mx = dx > dy ? dx : dy;
    mx = mx > dz ? mx : dz;
    ex = ey = ez = -((mx + 1) >> 1);
    k = 0;
    kend = mx;
  }
  // walk only cells [k0, k1) of the ray: cell k0 and its error terms by the
  // closed form (n steps along an axis after k cells: n = floor((2k|d| +
  // mx) / (2mx)), error k|d| - n mx), the same state stepping from 0 reaches
  BXG_HD void seek(int32_t k0, int32_t k1) {
    int32_t nx, ny, nz;
    steps(k0, nx, ny, nz);
    cx += sx * nx;
    cy += sy * ny;
    cz += sz * nz;
    const int32_t h = (mx + 1) >> 1;
    ex = (int32_t)((int64_t)k0 * dx - (int64_t)nx * mx) - h;
    ey = (int32_t)((int64_t)k0 * dy - (int64_t)ny * mx) - h;
    ez = (int32_t)((int64_t)k0 * dz - (int64_t)nz * mx) - h;
    k = k0;
    kend = k1;
  }
  // steps the walk has taken along each axis when it reaches cell k0 (mx > 0)
  BXG_HD void steps(int32_t k0, int32_t& nx, int32_t& ny, int32_t& nz) const {
    if (mx <= kRay32) {  // 2 k |d| + mx < 2^31 + 2^15
      const uint32_t m2 = 2u * (uint32_t)mx, k2 = 2u * (uint32_t)k0;
      nx = (int32_t)((k2 * (uint32_t)dx + (uint32_t)mx) / m2);
      ny = (int32_t)((k2 * (uint32_t)dy + (uint32_t)mx) / m2);
      nz = (int32_t)((k2 * (uint32_t)dz + (uint32_t)mx) / m2);
      return;
    }
    const int64_t m2 = 2 * (int64_t)mx;
    nx = (int32_t)((2 * (int64_t)k0 * dx + mx) / m2);
    ny = (int32_t)((2 * (int64_t)k0 * dy + mx) / m2);
    nz = (int32_t)((2 * (int64_t)k0 * dz + mx) / m2);
  }
  BXG_HD bool done() const { return k >= kend; }
  BXG_HD void cell(int32_t& x, int32_t& y, int32_t& z) const {
    x = cx;
    y = cy;
    z = cz;
  }
};

// Advance a walk through the cells of its current leaf (2^lb cells a side),
// at most kRun of them, recording their leaf-local indices; returns how many.
// Slots past the run hold the run's first index, so that every slot names a
// cell of the leaf and a load from it needs no branch.
//
// Per axis the walk keeps T = (steps the axis may still take inside the leaf)
// + (cells advanced so far): a step along the axis leaves T unchanged, a cell
// without one adds 1, and cell k + j is in the leaf iff T >= j on every
// axis.  The local index moves by the axis's stride on a step.  With the
// error terms biased by h, the step test is the sign of e, so one cell costs
// a few adds, shifts and masks an axis and no compare-and-select chain.
BXG_HD uint32_t collect_cells(RayWalk& w, uint32_t lb, uint32_t li[kRun]) {
  const int32_t lm = (1 << lb) - 1;
  const int32_t ux = w.cx & lm, uy = w.cy & lm, uz = w.cz & lm;
  const int32_t tx0 = w.sx > 0 ? lm - ux : ux;
  const int32_t ty0 = w.sy > 0 ? lm - uy : uy;
  const int32_t tz0 = w.sz > 0 ? lm - uz : uz;
  // a step's stride in the leaf-local index, negated (added where the axis
  // does not step, after all three were added)
  const int32_t qx = w.sx, qy = w.sy * (1 << lb), qz = w.sz * (1 << (2 * lb));
  const int32_t qall = qx + qy + qz;
  int32_t idx = ux | (uy << lb) | (uz << (2 * lb));
  const uint32_t l0 = (uint32_t)idx;
  int32_t ex = w.ex, ey = w.ey, ez = w.ez;
  int32_t tx = tx0, ty = ty0, tz = tz0;
  const int32_t rem = w.kend - w.k;
  const int32_t mx = w.mx, dx = w.dx, dy = w.dy, dz = w.dz;
  uint32_t n = 0;
#pragma unroll
  for (int j = 0; j < kRun; ++j) {
    int32_t t = tx < ty ? tx : ty;
    t = t < tz ? t : tz;
    const bool in = (j < rem) & (t >= j);
    li[j] = in ? (uint32_t)idx : l0;
    if (in) {
      n = (uint32_t)j + 1u;
      ex += dx;
      ey += dy;
      ez += dz;
      const int32_t nx = ex >> 31, ny = ey >> 31, nz = ez >> 31;  // -1: no step
      ex -= ~nx & mx;
      ey -= ~ny & mx;
      ez -= ~nz & mx;
      tx -= nx;
      ty -= ny;
      tz -= nz;
      idx += qall - (nx & qx) - (ny & qy) - (nz & qz);
    }
  }
  // steps taken along an axis: n less the cells without one (T's growth)
  w.cx += w.sx * ((int32_t)n - (tx - tx0));
  w.cy += w.sy * ((int32_t)n - (ty - ty0));
  w.cz += w.sz * ((int32_t)n - (tz - tz0));
  w.ex = ex;
  w.ey = ey;
  w.ez = ez;
  w.k += (int32_t)n;
  return n;
}

// The same walk for rays of at most kRay32 cells, with the error terms of two
// axes in the 16-bit halves of a word.  The axis of the longest step (d)
// steps at every cell and needs none; the others are a and b, each with
//   f = -1 - e   (below 0 after a cell: the axis steps),
//   S            (steps it may still take inside the leaf).
// A cell of the leaf has index K - Td qd - Sa qa - Sb qb + j qd, with q an
// axis's signed stride, Td the leaf's steps left along d at the run's first
// cell and K the sum of the ends of the rising axes: one dot product.  About 13
// instructions a cell, 26 in the 32-bit walk; no branch, as a run that has
// ended keeps f >= 0 (with branches a 100k-point room took 44 us for 25).  The
// walk that only marks cells is bound by the vector units (64 first scans 1.55
// -> 1.43 ms), the others less (a LiDAR scan of a map in use 2.5 %, 64
// re-inserted scans 2 %).
typedef int16_t i16x2 __attribute__((vector_size(4)));
struct RayWalk16 {
  int32_t cd, ca, cb;  // cell k along the permuted axes
  int32_t nd, na, nb;  // -1 where the axis falls, 0 where it rises
  i16x2 f, D, M;       // error terms, |d| of a and b, mx twice
  int32_t qd, K;
  i16x2 q;             // -qa, -qb
  int32_t k, kend;
  int32_t my, mz;      // -1 where d is y, z; a and b are y and z, with x in d's place
  BXG_HD void init(const RayWalk& w, uint32_t lb) {
    const int32_t lm = (1 << lb) - 1;
    mz = w.mx != w.dx && w.mx != w.dy ? -1 : 0;
    my = w.mx != w.dx ? ~mz : 0;
    cd = w.cx, ca = w.cy, cb = w.cz;
    swap(cd, ca, cb);
    int32_t sd = w.sx, sa = w.sy, sb = w.sz, hd = 0, ha = (int32_t)lb, hb = 2 * (int32_t)lb;
    int32_t ed = w.ex, ea = w.ey, eb = w.ez, dd = w.dx, da = w.dy, db = w.dz;
    swap(sd, sa, sb);
    swap(hd, ha, hb);
    swap(ed, ea, eb);
    swap(dd, da, db);
    nd = sd >> 31;
    na = sa >> 31;
    nb = sb >> 31;
    f = i16x2{(int16_t)~ea, (int16_t)~eb};
    D = i16x2{(int16_t)da, (int16_t)db};
    M = i16x2{(int16_t)w.mx, (int16_t)w.mx};
    qd = sd * (1 << hd);
    q = i16x2{(int16_t)(-sa * (1 << ha)), (int16_t)(-sb * (1 << hb))};
    K = (nd ? 0 : lm << hd) + (na ? 0 : lm << ha) + (nb ? 0 : lm << hb);
    k = w.k;
    kend = w.kend;
  }
  BXG_HD bool done() const { return k >= kend; }
  // x, y, z to d, a, b and back: x changes places with d
  BXG_HD void swap(int32_t& x, int32_t& y, int32_t& z) const {
    const int32_t ty = (x ^ y) & my, tz = (x ^ z) & mz;
    x ^= ty ^ tz;
    y ^= ty;
    z ^= tz;
  }
  BXG_HD void cell(int32_t& x, int32_t& y, int32_t& z) const {
    x = cd, y = ca, z = cb;
    swap(x, y, z);
  }
  BXG_HD static int32_t dot(i16x2 a, i16x2 b, int32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sdot2(a, b, c, false);
#else
    return c + (int32_t)a[0] * b[0] + (int32_t)a[1] * b[1];
#endif
  }
};

// collect_cells for a RayWalk16
BXG_HD uint32_t collect_cells(RayWalk16& w, uint32_t lb, uint32_t li[kRun]) {
  const int32_t lm = (1 << lb) - 1;
  const int32_t td = ~(w.cd ^ w.nd) & lm, ta = ~(w.ca ^ w.na) & lm, tb = ~(w.cb ^ w.nb) & lm;
  const int32_t rem = w.kend - w.k, most = rem < td + 1 ? rem : td + 1;
  i16x2 S = {(int16_t)ta, (int16_t)tb};
  i16x2 f = w.f;
  int32_t base = w.K - td * w.qd;
  const uint32_t l0 = (uint32_t)RayWalk16::dot(S, w.q, base);
  uint32_t n = 0;
#pragma unroll
  for (int j = 0; j < kRun; ++j) {
    uint32_t left;
    __builtin_memcpy(&left, &S, 4);
    const bool in = (j < most) & ((left & 0x80008000u) == 0);
    const uint32_t at = (uint32_t)RayWalk16::dot(S, w.q, base);
    li[j] = in ? at : l0;
    n += in ? 1u : 0u;
    base += w.qd;
    f -= in ? w.D : i16x2{0, 0};  // past the run f stays >= 0: no axis steps
    const i16x2 s = f >> 15;      // -1: the axis steps
    f += s & w.M;
    S += s;
  }
  w.f = f;
  const int32_t ma = ta - S[0], mb = tb - S[1];  // steps taken
  w.cd += ((int32_t)n ^ w.nd) - w.nd;
  w.ca += (ma ^ w.na) - w.na;
  w.cb += (mb ^ w.nb) - w.nb;
  w.k += (int32_t)n;
  return n;
}

// The leaves a ray's cells [k, kend) lie in, one leaf per step, without
// visiting the cells, as inner cells of their roots.  Along an axis with
// |d| > 0 the ray takes its n-th step at cell ceil((2n - 1) m / (2|d|)) (the
// inverse of the closed form), so the cell at which it enters the leaf N axis
// steps away is that value for N; the next boundary is L steps further, which
// adds floor(L m / |d|) and a remainder to the quotient, so after the set-up
// (a few divisions a ray) each leaf costs additions and compares only.  Axes
// crossing at the same cell move the ray diagonally, into one leaf.  Same
// leaves, in the same order, as the cell walk.
//
// The leaf pass of long winner lists is bound by the vector units (with a
// branch an axis and three coordinates 345 M wavefront instructions, 4 cycles
// each, for 64 scans), so a step is short: no branch an axis, and a leaf's
// place in its root is one packed word (64 re-inserted scans 505 -> 390 us,
// a LiDAR scan of a map in use 43 -> 37).
struct LeafWalk {
  uint32_t kx, ky, kz;  // cell at which the ray enters the next leaf along each axis
  uint32_t ex, ey, ez;  // k * 2|d| less the exact crossing (2N - 1) m, below 2|d|
  uint32_t Qx, Qy, Qz, Rx, Ry, Rz;  // per further leaf: floor(L m / |d|), 2 (L m mod |d|)
  uint32_t bx, by, bz;  // 2|d|
  uint32_t sx, sy, sz;  // a step of one leaf along each axis in p
  // Place of the current leaf in its root: below bit kLow the inner cell + 2^13
  // (its step out of the root neither borrows nor carries past kLow), above it
  // kField bits an axis, index + 2^ib, which leaves [2^ib, 2^(ib+1)) with a
  // step out of the root.
  uint32_t p;
  int32_t rx, ry, rz;  // origin of the root
  int32_t k, kend;
  static constexpr uint32_t kNever = 0xFFFFFFFFu;
  static constexpr uint32_t kField = 6, kLow = 14;
  static constexpr uint32_t kBit = 63u;  // of the inner cell in its word
  static constexpr uint32_t kX = kLow, kY = kLow + kField, kZ = kLow + 2 * kField;
  static constexpr uint32_t kOnes = (1u << kX) | (1u << kY) | (1u << kZ);
  BXG_HD static void axis(int32_t c, int32_t s, int32_t d, int32_t n, int32_t m, uint32_t L, uint32_t& kc,
                          uint32_t& e, uint32_t& Q, uint32_t& R, uint32_t& b) {
    const int32_t lm = (int32_t)L - 1;
    b = 2u * (uint32_t)(d > 0 ? d : 1);
    if (d == 0) {
      kc = kNever;
      e = Q = R = 0;
      return;
    }
    // axis steps from the origin to the first cell of the next leaf
    const int64_t N = (int64_t)n + (s > 0 ? (int64_t)L - (c & lm) : (int64_t)(c & lm) + 1);
    uint32_t q, r;  // (2N - 1) m = q * 2|d| + r
    if (m <= kRay32) {  // in 32 bits: (2N - 1) m < 2^32
      const uint32_t A = (uint32_t)(2 * N - 1) * (uint32_t)m, LM = L * (uint32_t)m;
      q = A / b;
      r = A - q * b;
      Q = LM / (uint32_t)d;
      R = 2u * (LM - Q * (uint32_t)d);
    } else {
      const uint64_t A = (uint64_t)(2 * N - 1) * (uint64_t)m;
      const uint64_t q64 = A / b;
      const uint64_t LM = (uint64_t)L * (uint64_t)m;
      const uint64_t Q64 = LM / (uint64_t)d;
      // quotients past 2^30 are beyond any ray (kend < 2^30): such an axis
      // never crosses again, and the sums of next() stay below 2^32
      q = (uint32_t)(q64 < (1ull << 30) ? q64 : (1ull << 30));
      r = (uint32_t)(A - q64 * b);
      Q = (uint32_t)(Q64 < (1ull << 30) ? Q64 : (1ull << 30));
      R = 2u * (uint32_t)(LM - Q64 * (uint64_t)d);
    }
    kc = q + (r > 0 ? 1u : 0u);
    e = r > 0 ? b - r : 0u;
  }
  // the leaf of cell w.k, walking cells [w.k, w.kend) of w's ray
  BXG_HD void init(const RayWalk& w, uint32_t lb, uint32_t ib) {
    const uint32_t L = 1u << lb, im = (1u << ib) - 1u;
    const int32_t rmask = ~((1 << (lb + ib)) - 1);
    k = w.k;
    kend = w.kend;
    // axis steps already taken at cell k (none at k = 0)
    int32_t nx = 0, ny = 0, nz = 0;
    if (k) w.steps(k, nx, ny, nz);
    axis(w.cx, w.sx, w.dx, nx, w.mx, L, kx, ex, Qx, Rx, bx);
    axis(w.cy, w.sy, w.dy, ny, w.mx, L, ky, ey, Qy, Ry, by);
    axis(w.cz, w.sz, w.dz, nz, w.mx, L, kz, ez, Qz, Rz, bz);
    sx = (uint32_t)w.sx * ((1u << kX) + 1u);
    sy = (uint32_t)w.sy * ((1u << kY) + (1u << ib));
    sz = (uint32_t)w.sz * ((1u << kZ) + (1u << 2 * ib));
    rx = w.cx & rmask;
    ry = w.cy & rmask;
    rz = w.cz & rmask;
    place(((uint32_t)(w.cx >> lb) & im) + im + 1u, ((uint32_t)(w.cy >> lb) & im) + im + 1u,
          ((uint32_t)(w.cz >> lb) & im) + im + 1u, ib);
  }
  BXG_HD void place(uint32_t fx, uint32_t fy, uint32_t fz, uint32_t ib) {
    const uint32_t im = (1u << ib) - 1u;
    p = (fx << kX) | (fy << kY) | (fz << kZ) | (1u << (kLow - 1)) | (fx & im) | ((fy & im) << ib) |
        ((fz & im) << 2 * ib);
  }
  BXG_HD bool done() const { return k >= kend; }
  // whether the current leaf is in the root (rx, ry, rz): (p & inside_mask) ==
  // inside_word.  With the word of the inner cell (its bits 6 and up) in both,
  // whether it is in that word too.
  BXG_HD static uint32_t inside_mask(uint32_t ib) { return ((1u << kField) - (1u << ib)) * kOnes; }
  BXG_HD static uint32_t inside_word(uint32_t ib) { return kOnes << ib; }
  BXG_HD static uint32_t word_mask(uint32_t ib) { return ((1u << 3 * ib) - 1u) & ~63u; }
  BXG_HD bool inside(uint32_t ib) const { return (p & inside_mask(ib)) == inside_word(ib); }
  BXG_HD static uint32_t turn(uint32_t f, int32_t& r, uint32_t one, int32_t size) {
    f &= (1u << kField) - 1u;
    if (f < one) {
      r -= size;
      return f + one;
    }
    if (f >= 2u * one) {
      r += size;
      return f - one;
    }
    return f;
  }
  // after a step out of the root: the root the current leaf is in
  BXG_HD void enter(uint32_t lb, uint32_t ib) {
    const uint32_t fx = turn(p >> kX, rx, 1u << ib, 1 << (lb + ib));
    const uint32_t fy = turn(p >> kY, ry, 1u << ib, 1 << (lb + ib));
    const uint32_t fz = turn(p >> kZ, rz, 1u << ib, 1 << (lb + ib));
    place(fx, fy, fz, ib);
  }
  // inner cell of the current leaf, which is inside the root
  BXG_HD uint32_t cell(uint32_t ib) const { return p & ((1u << 3 * ib) - 1u); }
  BXG_HD static void cross(bool at, uint32_t& kc, uint32_t& e, uint32_t& p, uint32_t Q, uint32_t R, uint32_t b,
                           uint32_t s) {
    const uint32_t r = at ? R : 0u;
    const bool more = e < r;
    kc += (at ? Q : 0u) + (more ? 1u : 0u);
    e = e - r + (more ? b : 0u);
    p += at ? s : 0u;
  }
  // move to the next leaf, or to kend: the ray is done then, and takes no
  // further step
  BXG_HD void next() {
    uint32_t kn = kx < ky ? kx : ky;
    kn = kn < kz ? kn : kz;
    cross(kx == kn, kx, ex, p, Qx, Rx, bx, sx);
    cross(ky == kn, ky, ey, p, Qy, Ry, by, sy);
    cross(kz == kn, kz, ez, p, Qz, Rz, bz, sz);
    k = (int32_t)(kn < (uint32_t)kend ? kn : (uint32_t)kend);
  }
};

// The tasks of a walk over a list of nb batches of 64 rays by a number of
// wavefronts spread over the XCDs (workgroups go round them): the wave-th
// wavefront of an XCD takes the tasks j = wave, wave + (the XCD's wavefronts), ...
// while task() gives one.
//
// A short list, with more wavefronts than batches: each ray is cut into up to
// 32 segments (2,001 points: update pass 25 us with 8, 20 with 16, 16 with 32),
// and a task is one segment of a batch.  With batches enough for 8 groups an XCD
// or more, the tasks of a group of up to 8 batches follow each other on one XCD,
// segment by segment, so that its L2 sees neighbours at one distance from the
// sensor.  With fewer, the segments of each batch go round the XCDs: kept on one
// each, those of one batch, a scan of up to 64 points, had an eighth of the
// wavefronts to themselves while the others had none (10 points, 50 m: 129 us a
// call, 60 so; 100: 103, 61; 1,000 to 8,000 points the same).  A long list: one
// contiguous part of it an XCD (a map's rays stay on one XCD or two), the rays
// walked whole.
constexpr uint32_t kXcds = 8;
constexpr uint32_t kMaxSegLog = 5;  // at most 32 segments a ray
constexpr uint32_t kGroupLog = 3;   // batches side by side on one XCD in a short list
struct WalkPlan {
  uint32_t nb, lg, gl, per_xcd;
  BXG_HD WalkPlan(uint32_t batches, uint32_t wavefronts) : nb(batches), lg(0), gl(kGroupLog) {
    while (lg < kMaxSegLog && ((uint64_t)nb << (lg + 1)) <= wavefronts) ++lg;
    while (gl > 0 && (nb >> gl) < 8u * kXcds) --gl;
    per_xcd = (nb + kXcds - 1) / kXcds;
  }
  BXG_HD bool whole() const { return lg == 0; }
  // task j of an XCD; false past its last one.  A batch at or past nb: nothing to do.
  BXG_HD bool task(uint32_t j, uint32_t xcd, uint32_t& batch, uint32_t& seg) const {
    seg = 0;
    if (whole()) {
      batch = xcd * per_xcd + j;
      return j < per_xcd;
    }
    if (gl == 0) {
      const uint32_t t = j * kXcds + xcd;
      batch = t >> lg;
      seg = t & ((1u << lg) - 1u);
      return batch < nb;
    }
    const uint32_t group = (j >> (gl + lg)) * kXcds + xcd;
    batch = (group << gl) + (j & ((1u << gl) - 1u));
    seg = (j >> gl) & ((1u << lg) - 1u);
    return (group << gl) < nb;
  }
};

}  // namespace bxg

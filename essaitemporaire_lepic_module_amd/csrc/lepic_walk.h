// lepic_walk.h -- which nodes or cells a thread of a bounded launch takes (host
// and device: tests/walk_check.cpp counts the visits on the host).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define LEPIC_HD __host__ __device__
#else
#define LEPIC_HD
#endif

// for (t; t < end; t += step).  I: int64_t, or uint32_t (2 % of a periodic solve):
// a level has up to 2^31 - 1 nodes, and the step past its last node has to stay
// beyond end.  In an int it wraps to a negative number, which the loop takes for
// a node; in 32 unsigned bits it does not, for steps below 2^31.
template <class I>
struct WalkT {
  I t, end, step;
};
using NodeWalk = WalkT<int64_t>;

// Striding over all blocks.
template <class I = int64_t>
LEPIC_HD inline WalkT<I> walk_strided(int64_t nodes, int block, int blocks, int thread,
                                      int threads) {
  return {(I)((int64_t)block * threads + thread), (I)nodes, (I)((int64_t)blocks * threads)};
}

// The blocks of each of `groups` (the XCDs, which take blocks in turn) walk
// their own share of the nodes in order.
LEPIC_HD inline NodeWalk walk_grouped(int64_t nodes, int block, int blocks, int thread,
                                      int threads, int groups) {
  if (blocks % groups != 0) return walk_strided(nodes, block, blocks, thread, threads);
  const int64_t per = (nodes / groups + threads) / threads * threads, b = block % groups * per;
  return {b + (int64_t)(block / groups) * threads + thread, b + per < nodes ? b + per : nodes,
          (int64_t)(blocks / groups) * threads};
}

// Exact x / d for x, d < 2^32: m = ceil(2^64 / d) (2^64 / d for powers of
// two), q = high 64 bits of x * m.  x m / 2^64 exceeds x / d by less than
// x / 2^64 < 2^-32 <= 1/d, so the floor is exact.
struct UDiv {
  uint64_t m;
  uint32_t d;
};

inline UDiv make_udiv(uint32_t d) {
  UDiv u;
  u.d = d;
  u.m = d <= 1 ? 0 : (~0ull) / d + 1;
  return u;
}

LEPIC_HD inline uint32_t udiv(uint32_t x, const UDiv &u) {
#ifdef __HIP_DEVICE_COMPILE__
  return u.d <= 1 ? x : (uint32_t)__umul64hi((uint64_t)x, u.m);
#else
  return u.d <= 1 ? x : (uint32_t)(((unsigned __int128)x * u.m) >> 64);
#endif
}

// Bricks of cells dealt to the XCDs (the sort's place pass).  A brick is about
// what an XCD's CUs hold at once, longer in x the fewer lanes a cell takes (a row
// of 16 thin cells is less than a memory line): 16, 32 or 64 x 8 x 8 cells, cut to
// near equal extents (17 cells are two of 9 and 8, not 16 and 1) and, while the
// grid has fewer than 64, halved.  Of each group of 8 bricks every XCD takes one,
// turned by a hash of the group, so that a set in part of the box (a slab, a beam)
// is spread over all of them: with consecutive bricks on one XCD a slab of 13
// planes of 128^3 took 1205 us, now 298.
struct BrickPlan {
  int n[3], e[3];              // cells, and a brick's, per axis
  uint32_t cells, bricks;      // per brick, in all
  uint32_t tasks;              // cell numbers per XCD, those of no cell included
  UDiv d_cells, d_nb0, d_nb1, d_e0, d_e1;
};

constexpr int BRICK_XCDS = 8;

inline BrickPlan brick_plan(const int32_t n[3], int lanes) {
  int e[3] = {lanes <= 8 ? 64 : lanes <= 32 ? 32 : 16, 8, 8}, nb[3];
  auto cut = [&]() {
    for (int d = 0; d < 3; ++d) {
      nb[d] = (n[d] + e[d] - 1) / e[d];
      e[d] = (n[d] + nb[d] - 1) / nb[d];
      nb[d] = (n[d] + e[d] - 1) / e[d];
    }
  };
  for (cut(); (int64_t)nb[0] * nb[1] * nb[2] < 64 && e[0] * e[1] * e[2] > 1; cut()) {
    int d = 2;
    if (e[1] > e[d]) d = 1;
    if (e[0] > e[d]) d = 0;
    e[d] = (e[d] + 1) / 2;
  }
  BrickPlan b;
  for (int d = 0; d < 3; ++d) {
    b.n[d] = n[d];
    b.e[d] = e[d];
  }
  b.cells = (uint32_t)(e[0] * e[1] * e[2]);
  b.bricks = (uint32_t)nb[0] * (uint32_t)nb[1] * (uint32_t)nb[2];
  b.tasks = (b.bricks + BRICK_XCDS - 1) / BRICK_XCDS * b.cells;
  b.d_cells = make_udiv(b.cells);
  b.d_nb0 = make_udiv((uint32_t)nb[0]);
  b.d_nb1 = make_udiv((uint32_t)nb[1]);
  b.d_e0 = make_udiv((uint32_t)e[0]);
  b.d_e1 = make_udiv((uint32_t)e[1]);
  return b;
}

// The cell id of task t < tasks of an XCD, -1: none.
LEPIC_HD inline int brick_cell(const BrickPlan &b, uint32_t xcd, uint32_t t) {
  const uint32_t group = udiv(t, b.d_cells), l = t - group * b.cells;
  const uint32_t turn = (group * 2654435769u) >> 29;
  const uint32_t brick = group * BRICK_XCDS + ((xcd + turn) & (BRICK_XCDS - 1));
  const uint32_t by = udiv(brick, b.d_nb0), bz = udiv(by, b.d_nb1);
  const uint32_t ly = udiv(l, b.d_e0), lz = udiv(ly, b.d_e1);
  const int x = (int)((brick - by * b.d_nb0.d) * b.e[0] + (l - ly * b.d_e0.d)),
            y = (int)((by - bz * b.d_nb1.d) * b.e[1] + (ly - lz * b.d_e1.d)),
            z = (int)(bz * b.e[2] + lz);
  if (brick >= b.bricks || x >= b.n[0] || y >= b.n[1] || z >= b.n[2]) return -1;
  return x + b.n[0] * (y + b.n[1] * z);
}

// Blocks of the place pass per XCD, lanes per cell in blocks of `threads`: a wave
// per 64 / lanes tasks, up to BRICK_BLOCKS in all (2^28 threads: a launch takes
// fewer than 2^32), which then stride over the tasks.
constexpr uint32_t BRICK_BLOCKS = 1u << 20;

inline uint32_t brick_blocks(const BrickPlan &b, int lanes, int threads) {
  const uint64_t per = (uint64_t)(threads / lanes), want = (b.tasks + per - 1) / per;
  return (uint32_t)(want < BRICK_BLOCKS / BRICK_XCDS ? want : BRICK_BLOCKS / BRICK_XCDS);
}

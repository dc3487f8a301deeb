// lepic_walk.h -- which nodes a thread of a bounded launch takes (host and
// device: tests/walk_check.cpp counts the visits on the host).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define LEPIC_HD __host__ __device__
#else
#define LEPIC_HD
#endif

// for (t; t < end; t += step).  64-bit: a level has up to 2^31 - 1 nodes, and
// the step past its last node has to stay beyond end (in 32 bits it wraps to a
// negative number, which the loop takes for a node).
struct NodeWalk {
  int64_t t, end, step;
};

// Striding over all blocks.
LEPIC_HD inline NodeWalk walk_strided(int64_t nodes, int block, int blocks, int thread,
                                      int threads) {
  return {(int64_t)block * threads + thread, nodes, (int64_t)blocks * threads};
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

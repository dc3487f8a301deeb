// lepic_walk.h: every node once, none outside, up to the most nodes of a solve.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../essaitemporaire_lepic_module_amd/csrc/lepic_walk.h"

int main() {
  const int threads = 256, groups = 8;
  long bad = 0;
  // small sizes: each node exactly once
  for (int64_t nodes : {1, 255, 256, 257, 2047, 2048, 2049, 100003}) {
    for (int blocks : {1, 3, 8, 16, 24}) {
      for (int grouped = 0; grouped < 2; ++grouped) {
        std::vector<int> seen(nodes, 0);
        for (int b = 0; b < blocks; ++b)
          for (int t = 0; t < threads; ++t) {
            NodeWalk w = grouped ? walk_grouped(nodes, b, blocks, t, threads, groups)
                                 : walk_strided(nodes, b, blocks, t, threads);
            for (; w.t < w.end; w.t += w.step) {
              if (w.t < 0 || w.t >= nodes) ++bad;
              else ++seen[w.t];
            }
          }
        for (int v : seen) bad += v != 1;
      }
    }
  }
  // the largest levels: every visit in range and as many visits as nodes, over
  // all threads (a thread's visits counted from its first and last node)
  const int blocks = 1024;
  for (int64_t nodes : {(int64_t)INT32_MAX, (int64_t)2147458027, (int64_t)INT32_MAX - 262144}) {
    for (int grouped = 0; grouped < 2; ++grouped) {
      int64_t visits = 0;
      for (int b = 0; b < blocks; ++b)
        for (int t = 0; t < threads; ++t) {
          const NodeWalk w = grouped ? walk_grouped(nodes, b, blocks, t, threads, groups)
                                     : walk_strided(nodes, b, blocks, t, threads);
          if (w.t >= w.end) continue;
          const auto n = (w.end - w.t + w.step - 1) / w.step;
          // the loop's own type carries the step past the last node
          decltype(NodeWalk::t) past = (decltype(NodeWalk::t))(w.t + (n - 1) * w.step);
          past += w.step;
          if (w.t < 0 || w.end > nodes || past < w.end || past - w.step >= nodes) ++bad;
          visits += n;
        }
      bad += visits != nodes;
    }
  }
  std::printf("bad %ld\n", bad);
  return bad != 0;
}

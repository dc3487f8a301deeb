// lepic_walk.h: every node and every cell once, none outside, up to the largest
// grids; launches within what HIP takes; localised sets spread over the XCDs.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <functional>
#include <vector>

#include "../essaitemporaire_lepic_module_amd/csrc/lepic_walk.h"

namespace {

const int LANES[4] = {8, 16, 32, 64};

// Every cell once; the most an XCD has of the cells that fill() takes, over the mean.
double spread(const int32_t n[3], int lanes, const std::function<bool(int, int, int)> &fill,
              long &bad) {
  const BrickPlan b = brick_plan(n, lanes);
  std::vector<unsigned char> seen((size_t)n[0] * n[1] * n[2], 0);
  long load[BRICK_XCDS] = {}, total = 0;
  for (uint32_t x = 0; x < BRICK_XCDS; ++x)
    for (uint32_t t = 0; t < b.tasks; ++t) {
      const int c = brick_cell(b, x, t);
      if (c < 0) continue;
      if (c >= (int)seen.size() || seen[c]++) {
        ++bad;
        continue;
      }
      if (fill(c % n[0], c / n[0] % n[1], c / (n[0] * n[1]))) ++load[x], ++total;
    }
  for (unsigned char v : seen) bad += v != 1;
  return (double)*std::max_element(load, load + BRICK_XCDS) * BRICK_XCDS / (double)total;
}

long check_bricks() {
  long bad = 0;
  const int32_t grids[][3] = {{1, 1, 1},    {1, 1, 40},  {40, 1, 1},   {1, 40, 1},  {17, 9, 9},
                              {16, 8, 8},   {33, 17, 9}, {65, 64, 63}, {5, 3, 200}, {129, 7, 2},
                              {300, 300, 1}, {1, 257, 255}, {31, 2, 77}};
  const auto all = [](int, int, int) { return true; };
  for (const auto &n : grids)
    for (int lanes : LANES) {
      const double most = spread(n, lanes, all, bad);
      // a grid one cell past a brick: no XCD holds most of it
      if ((int64_t)n[0] * n[1] * n[2] >= 1000 && most > 1.5) {
        std::printf("%d %d %d lanes %d: %.2f\n", n[0], n[1], n[2], lanes, most);
        ++bad;
      }
    }
  const int32_t cube[3] = {128, 128, 128};
  const std::function<bool(int, int, int)> sets[] = {
      [](int x, int, int) { return x < 13; }, [](int, int y, int) { return y < 13; },
      [](int, int, int z) { return z < 13; }, [](int, int, int z) { return z >= 100; },
      [](int x, int y, int) { return (x - 64) * (x - 64) + (y - 64) * (y - 64) < 900; },
      [](int x, int y, int z) { return x < 64 && y < 64 && z < 64; }};
  for (const auto &f : sets)
    for (int lanes : LANES) {
      const double most = spread(cube, lanes, f, bad);
      if (most > 1.6) {
        std::printf("set %d lanes %d: %.2f\n", (int)(&f - sets), lanes, most);
        ++bad;
      }
    }
  // launches: fewer than 2^32 threads with the listed cells' blocks (1024 at most),
  // on the widest grids (2^31 nodes with their ghosts)
  const int32_t wide[][3] = {{4096, 4096, 1},   {1, 4096, 4096},  {4096, 1, 4096},
                             {134217000, 1, 1}, {1, 1, 134217000}, {23160, 23160, 1},
                             {1, 23160, 23160}, {1287, 1287, 1287}, {2, 20724, 20724}};
  for (const auto &n : wide)
    for (int lanes : LANES) {
      const BrickPlan b = brick_plan(n, lanes);
      const uint64_t threads = ((uint64_t)brick_blocks(b, lanes, 256) * BRICK_XCDS + 1024) * 256;
      const uint64_t cells = (uint64_t)n[0] * n[1] * n[2];
      const uint64_t tasks = (uint64_t)((b.bricks + 7) / 8) * b.cells;
      // a thread's last step past the tasks stays in 32 bits
      if (threads >= 1ull << 32 || tasks != b.tasks || tasks * 8 < cells ||
          tasks * 8 > cells + cells / 3 + 64 * 4096 || tasks + threads / 64 >= 1ull << 32) {
        std::printf("%d %d %d lanes %d: threads %llu tasks %llu\n", n[0], n[1], n[2], lanes,
                    (unsigned long long)threads, (unsigned long long)tasks);
        ++bad;
      }
      // the last tasks decode to cells of the grid
      for (uint32_t x = 0; x < BRICK_XCDS; ++x)
        for (uint32_t t = b.tasks - 1; t + 300 > b.tasks && t < b.tasks; --t) {
          const int c = brick_cell(b, x, t);
          bad += c < -1 || (c >= 0 && (uint64_t)c >= cells);
        }
    }
  return bad;
}

// The largest levels: every visit in range and as many visits as nodes, over all
// threads (a thread's visits counted from its first and last node).
template <class I>
long check_largest() {
  const int threads = 256, groups = 8, blocks = 1024;
  long bad = 0;
  for (int64_t nodes : {(int64_t)INT32_MAX, (int64_t)2147458027, (int64_t)INT32_MAX - 262144}) {
    for (int grouped = 0; grouped < (sizeof(I) == 8 ? 2 : 1); ++grouped) {
      int64_t visits = 0;
      for (int b = 0; b < blocks; ++b)
        for (int t = 0; t < threads; ++t) {
          WalkT<I> w;
          if (grouped) {
            const NodeWalk g = walk_grouped(nodes, b, blocks, t, threads, groups);
            w = {(I)g.t, (I)g.end, (I)g.step};
          } else {
            w = walk_strided<I>(nodes, b, blocks, t, threads);
          }
          if (w.t >= w.end) continue;
          const int64_t n = ((int64_t)w.end - w.t + w.step - 1) / w.step;
          // the loop's own type carries the step past the last node
          const I last = (I)(w.t + (I)(n - 1) * w.step), past = (I)(last + w.step);
          if ((int64_t)w.t < 0 || (int64_t)w.end > nodes || past < w.end || last >= w.end) ++bad;
          visits += n;
        }
      bad += visits != nodes;
    }
  }
  return bad;
}

}  // namespace

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
  bad += check_largest<int64_t>() + check_largest<uint32_t>();
  bad += check_bricks();
  std::printf("bad %ld\n", bad);
  return bad != 0;
}

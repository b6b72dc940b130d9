// Host-only: what a call that steps pays for its plan (madpac_amd/csrc/lbm_pair.hip), on lattices whose split
// into chunks takes the longest search.  Prints the microseconds of the slowest plan; needs no device.
#include <algorithm>
#include <chrono>
#include <cstdio>

#include "lbm_internal.h"

using namespace lbm;

int main() {
  const int sizes[][3] = {{64, 64, 64}, {8, 8, 8192}, {16, 16, 2048}, {64, 8, 4096}, {1, 1, 270000}, {512, 512, 512}};
  const int periodic[3] = {1, 1, 1};
  double slowest = 0.0;
  for (const auto& n : sizes)
    for (int bricks = 0; bricks < 2; bricks++) {
      const DenseGeom g = make_geom(n[0], n[1], n[2], periodic, bricks != 0, 8, true);
      const PairSplits splits = pair_splits(g);  // once per context
      double best = 1e9;
      for (int trial = 0; trial < 5; trial++) {
        const auto t0 = std::chrono::steady_clock::now();
        for (int k = 0; k < 200; k++) {
          PairGeom plan;
          const bool pairs = pair_plan(g, splits, 8, g.Nu, false, (k & 1) != 0, false, 0, &plan);
          if (pairs && (int64_t)plan.cz * plan.tz < g.nz) return 1;
        }
        best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 200);
      }
      slowest = std::max(slowest, best);
    }
  std::printf("%.3f\n", slowest);
  return 0;
}

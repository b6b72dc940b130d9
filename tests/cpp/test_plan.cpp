// Host-only: the plan of a run of steps (madpac_amd/csrc/lbm_pair.hip); needs no device.
//
// usage: test_plan cost
//   prints the microseconds of the slowest plan, on lattices whose split into chunks takes the longest search
//        test_plan nx ny nz element_bytes fp32_arithmetic fluid_cells extra walls open
//   prints 1 where the two-step kernel is chosen (rows, periodic), else 0
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "lbm_internal.h"

using namespace lbm;

namespace {
const int PERIODIC[3] = {1, 1, 1};

int cost() {
  const int sizes[][3] = {{64, 64, 64}, {8, 8, 8192}, {16, 16, 2048}, {64, 8, 4096}, {1, 1, 270000}, {512, 512, 512}};
  double slowest = 0.0;
  for (const auto& n : sizes)
    for (int bricks = 0; bricks < 2; bricks++) {
      const DenseGeom g = make_geom(n[0], n[1], n[2], PERIODIC, bricks != 0, 8, true);
      const PairSplits splits = pair_splits(g);  // once per context
      double best = 1e9;
      for (int trial = 0; trial < 5; trial++) {
        const auto t0 = std::chrono::steady_clock::now();
        for (int k = 0; k < 200; k++) {
          PairGeom plan;
          const bool pairs = pair_plan(g, splits, 8, false, g.Nu, false, (k & 1) != 0, false, 0, &plan);
          if (pairs && (int64_t)plan.cz * plan.tz < g.nz) return 1;
        }
        best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 200);
      }
      slowest = std::max(slowest, best);
    }
  std::printf("%.3f\n", slowest);
  return 0;
}
}  // namespace

int main(int argc, char** argv) {
  if (argc == 2 && !std::strcmp(argv[1], "cost")) return cost();
  if (argc != 10) return 2;
  long long v[9];
  for (int k = 0; k < 9; k++) v[k] = std::atoll(argv[k + 1]);
  const DenseGeom g = make_geom((int)v[0], (int)v[1], (int)v[2], PERIODIC, false, (size_t)v[3], true);
  PairGeom plan;
  std::printf("%d\n", pair_plan(g, pair_splits(g), (size_t)v[3], v[4] != 0, v[5], v[6] != 0, v[7] != 0, v[8] != 0, 0, &plan));
  return 0;
}

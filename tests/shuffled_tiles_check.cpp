// build_tiles on elements in random order, on the CPU: tiles of consecutive elements then touch
// nodes all over the mesh, far more than a tile may, and have to end long before the asked size.
// Every plan keeps its capacities and owns every node once.  Exit status 1 on a failure.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>

#include "dendro_hip.h"
#include "host/octree.hpp"

using namespace dgh;

int main() {
  std::vector<double> pts(3 * 300000);
  if (dgh_points_generate(1, 300000, 7, 31, pts.data()) != 0) return 2;
  DALevel da;
  build_da(octree_from_points(pts.data(), 300000, 10, 1, true), 10, da);
  const uint32_t E = da.n_elem, N = da.n_node;
  std::vector<uint32_t> o(E), nl(size_t(E) * 8);
  std::iota(o.begin(), o.end(), 0u);
  std::shuffle(o.begin(), o.end(), std::mt19937(3));
  std::vector<uint8_t> child(E), hn(E), lev(E);
  for (uint32_t e = 0; e < E; ++e) {
    std::copy_n(&da.nlist[size_t(o[e]) * 8], 8, &nl[size_t(e) * 8]);
    child[e] = da.child[o[e]];
    hn[e] = da.hnmask[o[e]];
    lev[e] = da.lev[o[e]];
  }
  int failures = 0;
  struct { uint32_t T, budget, own_cap; } cases[] = {
      {64, 5056, 2048}, {192, 5056, 2048}, {621, 5056, 2048}, {1200, 5056, 2048}, {2048, 5056, 2048},   // 512 threads
      {700, 2496, 1024}, {3000, 10176, 4096},                                                           // 256, 1024
      {768, 3360, 1024}};                                                                               // elasticity
  for (const auto& c : cases) {
    TilePlan p;
    try {
      build_tiles(E, N, nl.data(), child.data(), hn.data(), lev.data(), c.T, p, c.budget, c.own_cap);
    } catch (const Error& e) {
      std::printf("FAIL T=%u budget=%u: %s\n", c.T, c.budget, e.what());
      ++failures;
      continue;
    }
    std::vector<int> owned(N, 0);
    for (const TileRec& t : p.tiles)
      for (uint32_t i = 0; i < t.n_own; ++i) owned[p.node_tab[t.node_off + i]]++;
    const bool ok = p.max_own <= c.own_cap && p.max_touch <= c.budget - c.own_cap &&
                    std::all_of(owned.begin(), owned.end(), [](int n) { return n == 1; });
    std::printf("%s T=%u budget=%u own_cap=%u: E=%u tiles=%zu max_own=%u max_touch=%u\n", ok ? "ok" : "FAIL", c.T, c.budget,
                c.own_cap, E, p.tiles.size(), p.max_own, p.max_touch);
    failures += !ok;
  }
  std::printf("%s (%d failures)\n", failures ? "FAILED" : "OK", failures);
  return failures ? 1 : 0;
}

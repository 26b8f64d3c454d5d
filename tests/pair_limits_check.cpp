// plan_pairs under its limits, on the CPU: the first tile size is max(32, E/256), every plan it accepts
// keeps within the limits and stores every node once, limits below one neighbourhood refuse the level
// (single sweeps then) and leave no plan behind.  Exit status 1 on a failure.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "dendro_hip.h"
#include "host/octree.hpp"

using namespace dgh;

static int failures = 0;
static void check(bool ok, const char* what, uint32_t at) {
  if (!ok && failures++ < 10) std::printf("FAIL limit %u: %s\n", at, what);
}

int main() {
  std::vector<double> pts(3 * 3000);
  if (dgh_points_generate(1, 3000, 7, 31, pts.data()) != 0) return 2;
  DALevel da;
  build_da(octree_from_points(pts.data(), 3000, 9, 1, true), 9, da);
  const uint32_t E = da.n_elem, N = da.n_node;
  auto plan = [&](uint32_t max_touch, uint32_t max_own, TilePlan& p) {
    return plan_pairs(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), max_touch, max_own, p);
  };
  TilePlan p;
  check(plan(N, N, p) && p.tile_elems == std::max(32u, E / 256u), "first size", N);
  const uint32_t touch0 = p.max_touch, own0 = p.max_own;
  uint32_t accepted = 0, refused = 0, smaller = 0;
  for (uint32_t lim = touch0 + 1; lim > 8; lim = lim * 3 / 4)
    for (int which = 0; which < 2; ++which) {
      TilePlan q;
      const bool ok = which ? plan(N, std::min(lim, own0), q) : plan(lim, N, q);
      if (!ok) {
        ++refused;
        check(q.tiles.empty() && q.rec_elem.empty(), "a refused plan is empty", lim);
        continue;
      }
      ++accepted;
      smaller += q.tile_elems < 32;
      check((which ? q.max_own : q.max_touch) <= lim, "within the limit", lim);
      std::vector<int> stored(N, 0);
      for (const TileRec& t : q.tiles)
        for (uint32_t i = 0; i < t.n_own2; ++i) stored[q.node_tab[t.node_off + i]]++;
      for (uint32_t v = 0; v < N; ++v) check(stored[v] == 1, "a node not stored once", lim);
    }
  check(accepted && refused && smaller, "limits that accept, shrink and refuse", 0);
  std::printf("E=%u N=%u first size: touched<=%u updated<=%u; %u accepted (%u in smaller tiles), %u refused: %s\n", E, N, touch0,
              own0, accepted, smaller, refused, failures ? "FAILED" : "OK");
  return failures ? 1 : 0;
}

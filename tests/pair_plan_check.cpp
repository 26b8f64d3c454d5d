// Contract of the two-sweep tile builder (build_pair_tiles), checked on the CPU.  The kernel that
// runs two sweeps on a tile relies on:
//   - every node being stored by exactly one tile, first in its node list (n_own2 of them);
//   - the first n_elem2 records being all elements touching a stored node, each once, and their
//     nodes being the first n_own of the list;
//   - the n_elem records being all elements touching one of those n_own nodes, each once;
//   - record vertex ids naming the nodes in the order k ^ child.
// Usage: pair_plan_check kind npts depth   (exit status 1 on a failure)
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "dendro_hip.h"
#include "host/octree.hpp"

using namespace dgh;

static int failures = 0;
static void check(bool ok, const char* what, size_t t) {
  if (!ok && failures++ < 10) std::printf("FAIL tile %zu: %s\n", t, what);
}

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const uint64_t n = std::strtoull(argv[2], nullptr, 10);
  const uint32_t D = uint32_t(std::atoi(argv[3]));
  std::vector<double> pts(3 * n);
  if (dgh_points_generate(std::atoi(argv[1]), n, 7, 31, pts.data()) != 0) return 2;
  DALevel da;
  build_da(octree_from_points(pts.data(), n, D, 1, true), D, da);
  const uint32_t E = da.n_elem, N = da.n_node;
  std::vector<std::set<uint32_t>> touching(N);
  for (uint32_t e = 0; e < E; ++e)
    for (int k = 0; k < 8; ++k) touching[da.nlist[size_t(e) * 8 + k]].insert(e);
  for (uint32_t T : {1u, 32u, 100u, E + 5u}) {
    TilePlan p;
    build_pair_tiles(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), T, p);
    std::vector<int> stored(N, 0);
    for (size_t t = 0; t < p.tiles.size(); ++t) {
      const TileRec& tr = p.tiles[t];
      const uint32_t* nodes = p.node_tab.data() + tr.node_off;
      check(tr.n_own2 <= tr.n_own && tr.n_own <= tr.n_touch && tr.n_elem2 <= tr.n_elem, "counts", t);
      check(std::set<uint32_t>(nodes, nodes + tr.n_touch).size() == tr.n_touch, "a node listed twice", t);
      for (uint32_t i = 0; i < tr.n_own2; ++i) stored[nodes[i]]++;
      std::set<uint32_t> want2, want, got2, got;
      for (uint32_t i = 0; i < tr.n_own2; ++i) want2.insert(touching[nodes[i]].begin(), touching[nodes[i]].end());
      for (uint32_t i = 0; i < tr.n_own; ++i) want.insert(touching[nodes[i]].begin(), touching[nodes[i]].end());
      for (uint32_t r = 0; r < tr.n_elem; ++r) {
        const size_t g = size_t(tr.elem_off) + r;
        const uint32_t e = p.rec_elem[g];
        check(got.insert(e).second, "a record twice", t);
        if (r < tr.n_elem2) got2.insert(e);
        check((p.meta[g] >> 5) == da.lev[e], "level", t);
        for (int k = 0; k < 8; ++k) {
          const uint32_t l = p.lid[g * 8 + k];
          check(l < (r < tr.n_elem2 ? tr.n_own : tr.n_touch), "vertex id", t);
          check(nodes[l] == da.nlist[size_t(e) * 8 + (k ^ da.child[e])], "vertex node", t);
        }
      }
      // a tile without a stored node (its elements' nodes all belong to earlier tiles) keeps its own records
      check(tr.n_own2 == 0 || (std::includes(got2.begin(), got2.end(), want2.begin(), want2.end())), "second sweep", t);
      check(std::includes(got.begin(), got.end(), want.begin(), want.end()), "first sweep", t);
    }
    for (uint32_t v = 0; v < N; ++v) check(stored[v] == 1, "a node not stored once", v);
    std::printf("T=%u: E=%u N=%u tiles=%zu records=%zu first-sweep nodes<=%u touched<=%u\n", T, E, N, p.tiles.size(),
                p.rec_elem.size(), p.max_own, p.max_touch);
  }
  std::printf("%s (%d failures)\n", failures ? "FAILED" : "OK", failures);
  return failures ? 1 : 0;
}

// Owner-computes tiling of one mesh level for the atomic-free operator kernel.
//
// Elements are cut into tiles of consecutive Morton-ordered elements.  Every node is owned
// by exactly one tile (the tile of the first element, in Morton order, that has the node
// as a vertex).  A tile's record list holds its own elements plus the "halo" elements of
// other tiles that touch a node it owns; the kernel evaluates those records, accumulates
// the rows of owned nodes in LDS and stores each owned node once.  Inside a tile the
// records are sorted by class (child-0 type, then level) so that the wavefronts read mostly
// one stencil.
//
// Stencils are mirror images across child numbers: reflecting the axes on which child c
// has its bit set maps the element to child 0 and vertex k to vertex k^c, so
// K[c][t][k][j] = K[0][t'][k^c][j^c] where t' is the child-0 type of the reflected hanging
// mask.  A record therefore stores its vertex list permuted by k -> k^c and the child-0
// type t', and the kernel needs the 18 child-0 stencils only.
#include <algorithm>
#include <atomic>
#include <numeric>

#include "octree.hpp"
#include "workers.hpp"

namespace dgh {

static uint8_t mirror_mask(uint8_t mask, int c) {
  uint8_t m = 0;
  for (int k = 0; k < 8; ++k)
    if (mask & (1u << k)) m |= uint8_t(1u << (k ^ c));
  return m;
}

// Greedy cut: a tile grows one element at a time.  Adding element b makes it an own
// element (its nodes become touched) and makes it the owner of the nodes whose first
// touching element it is; every later element touching such a node joins the tile's halo
// (its nodes become touched too).  Owned and touched counts only grow, so the tile ends
// before the first element whose addition would exceed the budget or the element cap.
// With own_cap > 0 the owned nodes have a fixed capacity: a tile also ends before it owns
// more than own_cap nodes or touches more than budget - own_cap.
void tile_bounds(uint32_t E, uint32_t N, const uint32_t* nl, uint32_t T, uint32_t budget,
                 std::vector<uint32_t>& bounds, uint32_t own_cap) {
  bounds.clear();
  if (budget == 0) {
    for (uint32_t e = 0; e < E; e += T) bounds.push_back(e);
    bounds.push_back(E);
    return;
  }
  std::vector<uint32_t> first(N, 0xffffffffu);
  for (uint32_t e = 0; e < E; ++e)
    for (int k = 0; k < 8; ++k) {
      uint32_t& f = first[nl[size_t(e) * 8 + k]];
      if (f == 0xffffffffu) f = e;
    }
  // elements touching each node (CSR), in ascending element order
  std::vector<uint32_t> ptr(size_t(N) + 1, 0), adj(size_t(E) * 8);
  for (size_t i = 0; i < size_t(E) * 8; ++i) ptr[nl[i] + 1]++;
  for (uint32_t n = 0; n < N; ++n) ptr[n + 1] += ptr[n];
  {
    std::vector<uint32_t> fill(ptr.begin(), ptr.end() - 1);
    for (uint32_t e = 0; e < E; ++e)
      for (int k = 0; k < 8; ++k) adj[fill[nl[size_t(e) * 8 + k]]++] = e;
  }
  std::vector<uint32_t> nmark(N, 0), emark(E, 0);
  uint32_t stamp = 0;
  for (uint32_t a = 0; a < E;) {
    ++stamp;
    bounds.push_back(a);
    uint32_t own = 0, touch = 0, b = a;
    auto touch_elem = [&](uint32_t e) {
      if (emark[e] == stamp) return;
      emark[e] = stamp;
      for (int k = 0; k < 8; ++k) {
        const uint32_t n = nl[size_t(e) * 8 + k];
        if (nmark[n] != stamp) {
          nmark[n] = stamp;
          ++touch;
        }
      }
    };
    for (; b < E && b - a < T; ++b) {
      touch_elem(b);
      for (int k = 0; k < 8; ++k) {
        const uint32_t n = nl[size_t(b) * 8 + k];
        if (first[n] != b) continue;
        bool dup = false;   // a node listed twice in one element is owned once
        for (int q = 0; q < k; ++q) dup |= (nl[size_t(b) * 8 + q] == n);
        if (dup) continue;
        ++own;
        for (uint32_t p = ptr[n]; p < ptr[n + 1]; ++p)
          if (adj[p] > b) touch_elem(adj[p]);
      }
      if (touch > 65535u) break;
      if (own_cap ? (own > own_cap || own_cap + touch > budget) : (own + touch > budget)) break;
    }
    if (b == a) fail(DGH_ERR_ARG, "tile budget %u is smaller than one element's footprint", budget);
    a = b;
  }
  bounds.push_back(E);
}

static void build_from_bounds(uint32_t E, uint32_t N, const uint32_t* nl, const uint8_t* child, const uint8_t* hn,
                              const uint8_t* lev, const std::vector<uint32_t>& bounds, TilePlan& plan);

void build_tiles(uint32_t E, uint32_t N, const uint32_t* nl, const uint8_t* child, const uint8_t* hn,
                 const uint8_t* lev, uint32_t T, TilePlan& plan, uint32_t budget, uint32_t own_cap) {
  if (T < 64 || T > 16384) fail(DGH_ERR_ARG, "tile size %u out of range [64,16384]", T);
  if (own_cap && own_cap >= budget) fail(DGH_ERR_ARG, "owned-node capacity %u not below the budget %u", own_cap, budget);
  auto build = [&](const std::vector<uint32_t>& bounds) {
    plan = TilePlan();
    plan.tile_elems = T;
    plan.budget = budget;
    plan.own_cap = own_cap;
    build_from_bounds(E, N, nl, child, hn, lev, bounds, plan);
  };
  std::vector<uint32_t> bounds;
  // Tiles far below the budget are cut at T elements and checked afterwards: where none exceeds
  // its capacities the greedy cut is the same one (it ends a tile early only when its next element
  // would exceed them), and its node adjacency is most of the planning time (318k elements: 40 of
  // 60 ms).
  if (own_cap && T <= (budget - own_cap) / 2) {
    tile_bounds(E, N, nl, T, 0, bounds, 0);
    try {
      build(bounds);
      if (plan.max_own <= own_cap && plan.max_touch <= budget - own_cap) return;
    } catch (const Error& e) {
      if (e.code != DGH_ERR_ARG) throw;   // a tile beyond its vertex ids (elements in no spatial order)
    }
  }
  tile_bounds(E, N, nl, T, budget, bounds, own_cap);
  build(bounds);
}

// Child-0 type of every element's mirrored hanging mask.
static std::vector<uint8_t> element_types(uint32_t E, const uint8_t* child, const uint8_t* hn) {
  std::vector<int8_t> type_of(8 * 256);
  for (int c = 0; c < 8; ++c)
    for (int h = 0; h < 256; ++h) type_of[c * 256 + h] = int8_t(etype_of(0, mirror_mask(uint8_t(h), c)));
  std::vector<uint8_t> tp(E);
  for (uint32_t e = 0; e < E; ++e) {
    const int t0 = type_of[child[e] * 256 + hn[e]];
    if (t0 < 0) fail(DGH_ERR_MESH, "element %u: mirrored hanging mask is not a child-0 type", e);
    tp[e] = uint8_t(t0);
  }
  return tp;
}

// Orders a tile's records (of one sweep).  Classes: child-0 type, then level (uniform coefficients
// read one element matrix per (type, level) class); a counting sort keeps the Morton order inside a
// class.  cls_end (1024 entries) and sorted are scratch.
static void order_records(uint32_t* recs, size_t n, const uint8_t* tp, const uint8_t* lev,
                          std::vector<uint32_t>& cls_end, std::vector<uint32_t>& sorted) {
  auto cls = [&](uint32_t e) { return (uint32_t(tp[e]) << 5) | lev[e]; };
  std::fill(cls_end.begin(), cls_end.end(), 0u);
  for (size_t i = 0; i < n; ++i) ++cls_end[cls(recs[i])];
  uint32_t at = 0;
  for (uint32_t& c : cls_end) {
    const uint32_t m = c;
    c = at;
    at += m;
  }
  sorted.resize(n);
  for (size_t i = 0; i < n; ++i) sorted[cls_end[cls(recs[i])]++] = recs[i];
  // Inside each class, deal the Morton-ordered records round-robin over the class's
  // wavefronts: the 64 lanes of a wavefront then hold elements about n/64 apart, so
  // siblings (which share the parent-centre node after the mirror permutation) do
  // not collide on one LDS address in the same atomic instruction.
  size_t q = 0;
  for (size_t a = 0; a < sorted.size();) {
    const size_t b = cls_end[cls(sorted[a])], W = (b - a + 63) / 64;
    for (size_t w = 0; w < W; ++w)
      for (size_t i = a + w; i < b; i += W) recs[q++] = sorted[i];
    a = b;
  }
}

// Joins the per-tile records, node lists and ids into the plan.
static void concatenate(const std::vector<std::vector<uint32_t>>& t_rec, const std::vector<std::vector<uint32_t>>& t_nodes,
                        const std::vector<std::vector<uint16_t>>& t_lid, const std::vector<uint8_t>& tp,
                        const uint8_t* lev, TilePlan& plan) {
  const uint32_t ntiles = uint32_t(plan.tiles.size());
  size_t R = 0, NT = 0;
  for (uint32_t t = 0; t < ntiles; ++t) {
    plan.tiles[t].elem_off = uint32_t(R);
    plan.tiles[t].node_off = uint32_t(NT);
    R += t_rec[t].size();
    NT += t_nodes[t].size();
    plan.max_touch = std::max(plan.max_touch, plan.tiles[t].n_touch);
    plan.max_own = std::max(plan.max_own, plan.tiles[t].n_own);
    plan.max_elem = std::max(plan.max_elem, plan.tiles[t].n_elem);
    plan.max_slots = std::max(plan.max_slots, plan.tiles[t].n_own + plan.tiles[t].n_touch);
  }
  if (R > 0xffffffffu || NT > 0xffffffffu) fail(DGH_ERR_ARG, "mesh too large for 32-bit tile offsets");
  plan.rec_elem.resize(R);
  plan.meta.resize(R);
  plan.lid.resize(R * 8);
  plan.node_tab.resize(NT);
  for (uint32_t t = 0; t < ntiles; ++t) {
    const size_t ro = plan.tiles[t].elem_off, no = plan.tiles[t].node_off;
    std::copy(t_rec[t].begin(), t_rec[t].end(), plan.rec_elem.begin() + ro);
    std::copy(t_lid[t].begin(), t_lid[t].end(), plan.lid.begin() + ro * 8);
    std::copy(t_nodes[t].begin(), t_nodes[t].end(), plan.node_tab.begin() + no);
    for (size_t r = 0; r < t_rec[t].size(); ++r) {
      const uint32_t e = t_rec[t][r];
      plan.meta[ro + r] = uint16_t(tp[e] | (uint16_t(lev[e]) << 5));
    }
  }
}

// Runs f(w, nt) on nt workers; worker w takes every nt-th tile from w on.
template <class F>
static void for_tiles(uint32_t ntiles, F f) {
  const unsigned nt = worker_count(ntiles, 16);   // a worker's start costs as much as a dozen small tiles
  run_workers(nt, [&](unsigned w) { f(w, nt); });
}

static void build_from_bounds(uint32_t E, uint32_t N, const uint32_t* nl, const uint8_t* child, const uint8_t* hn,
                              const uint8_t* lev, const std::vector<uint32_t>& bounds, TilePlan& plan) {
  const uint32_t ntiles = uint32_t(bounds.size() - 1);
  std::vector<uint32_t> tile_of(E);
  for (uint32_t t = 0; t < ntiles; ++t)
    for (uint32_t e = bounds[t]; e < bounds[t + 1]; ++e) tile_of[e] = t;
  // owner tile of every node: first touching element's tile
  std::vector<uint32_t> owner(N, 0xffffffffu);
  for (uint32_t e = 0; e < E; ++e)
    for (int k = 0; k < 8; ++k) {
      uint32_t& o = owner[nl[size_t(e) * 8 + k]];
      if (o == 0xffffffffu) o = tile_of[e];
    }
  for (uint32_t n = 0; n < N; ++n)
    if (owner[n] == 0xffffffffu) fail(DGH_ERR_MESH, "node %u is not a vertex of any element", n);
  // halo elements per tile
  std::vector<std::vector<uint32_t>> halo(ntiles);
  for (uint32_t e = 0; e < E; ++e) {
    const uint32_t te = tile_of[e];
    uint32_t seen[8];
    int ns = 0;
    for (int k = 0; k < 8; ++k) {
      const uint32_t o = owner[nl[size_t(e) * 8 + k]];
      if (o == te) continue;
      bool dup = false;
      for (int q = 0; q < ns; ++q) dup |= (seen[q] == o);
      if (!dup) {
        seen[ns++] = o;
        halo[o].push_back(e);
      }
    }
  }
  // owned nodes per tile (ascending)
  std::vector<uint32_t> own_cnt(ntiles + 1, 0);
  for (uint32_t n = 0; n < N; ++n) own_cnt[owner[n] + 1]++;
  for (uint32_t t = 0; t < ntiles; ++t) own_cnt[t + 1] += own_cnt[t];
  std::vector<uint32_t> owned(N);
  {
    std::vector<uint32_t> fillp(own_cnt.begin(), own_cnt.end() - 1);
    for (uint32_t n = 0; n < N; ++n) owned[fillp[owner[n]]++] = n;
  }
  const std::vector<uint8_t> tp = element_types(E, child, hn);   // child-0 type t'
  // per-tile records, built in parallel (each worker keeps a dense node -> local id map)
  plan.tiles.resize(ntiles);
  std::vector<std::vector<uint32_t>> t_rec(ntiles), t_nodes(ntiles);
  std::vector<std::vector<uint16_t>> t_lid(ntiles);
  for_tiles(ntiles, [&](unsigned w, unsigned nt) {
      std::vector<int32_t> lid_of(N, -1);
      std::vector<uint32_t> cls_end(1024), sorted;
      for (uint32_t t = w; t < ntiles; t += nt) {
        auto& recs = t_rec[t];
        const uint32_t e0 = bounds[t], e1 = bounds[t + 1];
        recs.resize(e1 - e0);
        std::iota(recs.begin(), recs.end(), e0);
        recs.insert(recs.end(), halo[t].begin(), halo[t].end());
        order_records(recs.data(), recs.size(), tp.data(), lev, cls_end, sorted);
        auto& nodes = t_nodes[t];
        nodes.assign(owned.begin() + own_cnt[t], owned.begin() + own_cnt[t + 1]);
        for (size_t i = 0; i < nodes.size(); ++i) lid_of[nodes[i]] = int32_t(i);
        const size_t n_own = nodes.size();
        std::vector<uint32_t> extra;
        for (uint32_t e : recs)
          for (int k = 0; k < 8; ++k) {
            const uint32_t n = nl[size_t(e) * 8 + k];
            if (lid_of[n] == -1) {   // not owned and not yet listed
              lid_of[n] = -2;
              extra.push_back(n);
            }
          }
        std::sort(extra.begin(), extra.end());
        for (size_t i = 0; i < extra.size(); ++i) lid_of[extra[i]] = int32_t(n_own + i);
        nodes.insert(nodes.end(), extra.begin(), extra.end());
        if (nodes.size() > 65535) fail(DGH_ERR_ARG, "a tile touches more than 65535 nodes; use a smaller tile size");
        auto& lids = t_lid[t];
        lids.resize(recs.size() * 8);
        for (size_t r = 0; r < recs.size(); ++r) {
          const uint32_t e = recs[r];
          const int c = child[e];
          for (int k = 0; k < 8; ++k) lids[r * 8 + k] = uint16_t(lid_of[nl[size_t(e) * 8 + (k ^ c)]]);
        }
        for (uint32_t n : nodes) lid_of[n] = -1;
        plan.tiles[t].n_own = uint32_t(n_own);
        plan.tiles[t].n_touch = uint32_t(nodes.size());
        plan.tiles[t].n_elem = uint32_t(recs.size());
      }
  });
  concatenate(t_rec, t_nodes, t_lid, tp, lev, plan);
}

bool build_pair_tiles(uint32_t E, uint32_t N, const uint32_t* nl, const uint8_t* child, const uint8_t* hn,
                      const uint8_t* lev, uint32_t T, TilePlan& plan, uint32_t max_touch, uint32_t max_own) {
  max_touch = std::min(max_touch, 65535u);   // 16-bit vertex ids
  std::atomic<bool> over{false};
  plan = TilePlan();
  plan.tile_elems = T;
  const uint32_t ntiles = (E + T - 1) / T;
  plan.tiles.resize(ntiles);
  const std::vector<uint8_t> tp = element_types(E, child, hn);
  // elements touching each node (CSR, ascending): the first one's tile owns the node
  std::vector<uint32_t> ptr(size_t(N) + 1, 0), adj(size_t(E) * 8);
  for (size_t i = 0; i < size_t(E) * 8; ++i) ptr[nl[i] + 1]++;
  for (uint32_t n = 0; n < N; ++n) ptr[n + 1] += ptr[n];
  {
    std::vector<uint32_t> fill(ptr.begin(), ptr.end() - 1);
    for (uint32_t e = 0; e < E; ++e)
      for (int k = 0; k < 8; ++k) adj[fill[nl[size_t(e) * 8 + k]]++] = e;
  }
  std::vector<std::vector<uint32_t>> t_rec(ntiles), t_nodes(ntiles);
  std::vector<std::vector<uint16_t>> t_lid(ntiles);
  for_tiles(ntiles, [&](unsigned w, unsigned nt) {
    std::vector<int32_t> lid_of(N, -1);
    std::vector<uint32_t> emark(E, 0), cls_end(1024), sorted;
    for (uint32_t t = w; t < ntiles && !over.load(std::memory_order_relaxed); t += nt) {
      const uint32_t e0 = t * T, e1 = std::min(E, e0 + T);
      auto& recs = t_rec[t];
      auto& nodes = t_nodes[t];
      auto add_elem = [&](uint32_t e) {
        if (emark[e] == t + 1) return;
        emark[e] = t + 1;
        recs.push_back(e);
      };
      // lists the nodes of recs[from, ...) not listed yet, ascending; owned: only those of tile t
      auto add_nodes = [&](size_t from, bool owned) {
        const size_t n0 = nodes.size();
        for (size_t r = from; r < recs.size(); ++r)
          for (int k = 0; k < 8; ++k) {
            const uint32_t n = nl[size_t(recs[r]) * 8 + k];
            if (lid_of[n] != -1 || (owned && adj[ptr[n]] / T != t)) continue;
            lid_of[n] = -2;
            nodes.push_back(n);
          }
        std::sort(nodes.begin() + n0, nodes.end());
        for (size_t i = n0; i < nodes.size(); ++i) lid_of[nodes[i]] = int32_t(i);
      };
      auto add_elems_of = [&](size_t from) {
        for (size_t i = from; i < nodes.size(); ++i)
          for (uint32_t p = ptr[nodes[i]]; p < ptr[nodes[i] + 1]; ++p) add_elem(adj[p]);
      };
      for (uint32_t e = e0; e < e1; ++e) add_elem(e);
      add_nodes(0, true);
      const size_t n_out = nodes.size();
      add_elems_of(0);
      const size_t r2 = recs.size();
      add_nodes(0, false);
      const size_t n1 = nodes.size();
      add_elems_of(n_out);
      add_nodes(r2, false);
      if (nodes.size() > max_touch || n1 > max_own) {
        over = true;
        return;
      }
      order_records(recs.data(), r2, tp.data(), lev, cls_end, sorted);
      order_records(recs.data() + r2, recs.size() - r2, tp.data(), lev, cls_end, sorted);
      auto& lids = t_lid[t];
      lids.resize(recs.size() * 8);
      for (size_t r = 0; r < recs.size(); ++r)
        for (int k = 0; k < 8; ++k) lids[r * 8 + k] = uint16_t(lid_of[nl[size_t(recs[r]) * 8 + (k ^ child[recs[r]])]]);
      for (uint32_t n : nodes) lid_of[n] = -1;
      TileRec& tr = plan.tiles[t];
      tr.n_own = uint32_t(n1);
      tr.n_touch = uint32_t(nodes.size());
      tr.n_elem = uint32_t(recs.size());
      tr.n_own2 = uint32_t(n_out);
      tr.n_elem2 = uint32_t(r2);
    }
  });
  if (over) return false;
  concatenate(t_rec, t_nodes, t_lid, tp, lev, plan);
  return true;
}

bool plan_pairs(uint32_t E, uint32_t N, const uint32_t* nl, const uint8_t* child, const uint8_t* hn,
                const uint8_t* lev, uint32_t max_touch, uint32_t max_own, TilePlan& plan) {
  for (uint32_t T = std::max(32u, E / 256u); T >= 8; T /= 2)
    if (build_pair_tiles(E, N, nl, child, hn, lev, T, plan, max_touch, max_own)) return true;
  plan = TilePlan();
  return false;
}

bool build_gather(uint32_t nrows, const uint32_t* rowptr, const uint32_t* col, const float* w, uint32_t B,
                  GatherPlan& plan) {
  const uint32_t nb = (nrows + B - 1) / B;
  std::vector<std::vector<uint32_t>> cols(nb);
  plan.ent.resize(rowptr[nrows]);
  std::vector<int> bad(16, 0);
  for_tiles(nb, [&](unsigned wk, unsigned nt) {
    // the block's columns in an open-addressed table of twice the most it may hold
    constexpr uint32_t HS = 2u << GATHER_BITS;
    std::vector<uint32_t> key(HS), owner(HS, 0xffffffffu), slot(HS);
    uint32_t b = wk;
    auto find = [&](uint32_t c) {
      uint32_t h = (c * 2654435761u) >> (31 - GATHER_BITS);
      while (owner[h] == b && key[h] != c) h = (h + 1) & (HS - 1);
      return h;
    };
    for (; b < nb && !bad[wk]; b += nt) {
      const uint32_t q0 = rowptr[b * B], q1 = rowptr[std::min(nrows, (b + 1) * B)];
      auto& l = cols[b];
      for (uint32_t q = q0; q < q1 && l.size() <= GATHER_MAX; ++q) {
        const uint32_t h = find(col[q]);
        if (owner[h] == b) continue;
        owner[h] = b;
        key[h] = col[q];
        l.push_back(col[q]);
      }
      if (l.size() > GATHER_MAX) {
        bad[wk] = 1;
        break;
      }
      std::sort(l.begin(), l.end());
      for (size_t i = 0; i < l.size(); ++i) slot[find(l[i])] = uint32_t(i);
      for (uint32_t q = q0; q < q1; ++q) {
        const double k = double(w[q]) * 32.0;
        if (!(k >= 1.0 && k <= 32.0 && k == double(int(k)))) bad[wk] = 1;
        plan.ent[q] = uint16_t((uint32_t(k - 1.0) << GATHER_BITS) | slot[find(col[q])]);
      }
    }
  });
  for (int e : bad)
    if (e) return false;
  plan.pitch = 1;
  for (const auto& l : cols) plan.pitch = std::max(plan.pitch, uint32_t(l.size()));
  plan.list.assign(size_t(nb) * plan.pitch, 0u);
  for (uint32_t b = 0; b < nb; ++b) {
    uint32_t* dst = plan.list.data() + size_t(b) * plan.pitch;
    std::copy(cols[b].begin(), cols[b].end(), dst);
    if (!cols[b].empty()) std::fill(dst + cols[b].size(), dst + plan.pitch, cols[b].back());
  }
  return true;
}

}  // namespace dgh

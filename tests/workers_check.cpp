// The host planners when the system gives them no thread or no memory: a share whose thread cannot be
// started is done all the same, with the same plan, and an allocation that fails in a worker reaches the
// caller as std::bad_alloc, as one on the calling thread does.  Exit status 1 on a failure (an
// uncaught exception ends the program by a signal).
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "dendro_hip.h"
#include "host/octree.hpp"

using namespace dgh;

static int threads_left = 1 << 30;   // threads that may still be started
static int started = 0;
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  if (threads_left <= 0) return EAGAIN;
  --threads_left;
  ++started;
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  return real(t, a, f, arg);
}

static bool starve = false;   // large allocations fail, except on the main thread
static const pthread_t main_thread = pthread_self();
void* operator new(size_t n) {
  if (starve && n > 4096 && !pthread_equal(pthread_self(), main_thread)) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static int failures = 0;
static void check(bool ok, const char* what) {
  if (!ok && failures++ < 10) std::printf("FAIL %s\n", what);
}
template <class T>
static bool same(const std::vector<T>& a, const std::vector<T>& b) {
  return a.size() == b.size() && std::memcmp(a.data(), b.data(), a.size() * sizeof(T)) == 0;
}

int main() {
  std::vector<double> pts(3 * 30000);
  if (dgh_points_generate(1, 30000, 7, 31, pts.data()) != 0) return 2;
  const std::vector<Oct> leaves = octree_from_points(pts.data(), 30000, 9, 1, true);
  DALevel da;
  build_da(leaves, 9, da);
  const uint32_t E = da.n_elem, N = da.n_node;
  std::vector<uint32_t> ptr(1, 0), col;   // a transfer-like sparse matrix
  std::vector<float> w;
  for (uint32_t i = 0; i < N; ++i) {
    for (uint32_t k = 0; k < 4; ++k) {
      col.push_back((i + k) / 3);
      w.push_back(0.25f);
    }
    ptr.push_back(uint32_t(col.size()));
  }
  auto plans = [&](TilePlan& t, TilePlan& p, GatherPlan& g, DALevel& d) {
    build_tiles(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), 64, t);
    build_pair_tiles(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), 64, p);
    check(build_gather(N, ptr.data(), col.data(), w.data(), 64, g), "gather accepted");
    build_da(leaves, 9, d);
  };
  TilePlan t0, p0;
  GatherPlan g0;
  DALevel d0;
  plans(t0, p0, g0, d0);
  const int all = started;
  std::printf("E=%u N=%u threads started: %d\n", E, N, all);
  if (all == 0) std::printf("one CPU: nothing runs on a thread here\n");
  for (int n : {0, 1, all / 2, all - 1}) {
    if (n < 0) continue;
    threads_left = n;
    TilePlan t, p;
    GatherPlan g;
    DALevel d;
    plans(t, p, g, d);
    check(same(t.rec_elem, t0.rec_elem) && same(t.lid, t0.lid) && same(t.node_tab, t0.node_tab), "tiles");
    check(same(p.rec_elem, p0.rec_elem) && same(p.lid, p0.lid) && same(p.node_tab, p0.node_tab), "pair tiles");
    check(same(g.ent, g0.ent) && same(g.list, g0.list), "gather");
    check(same(d.nlist, d0.nlist) && same(d.hnmask, d0.hnmask), "mesh");
  }
  threads_left = 1 << 30;
  for (int q = 0; q < 3 && all > 0; ++q) {
    TilePlan t;
    GatherPlan g;
    bool threw = false;
    starve = true;
    try {
      if (q == 0) build_tiles(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), 64, t);
      if (q == 1) build_pair_tiles(E, N, da.nlist.data(), da.child.data(), da.hnmask.data(), da.lev.data(), 64, t);
      if (q == 2) build_gather(N, ptr.data(), col.data(), w.data(), 64, g);
    } catch (const std::bad_alloc&) {
      threw = true;
    }
    starve = false;
    check(threw, "a failed allocation is reported");
  }
  std::printf("%s (%d failures)\n", failures ? "FAILED" : "OK", failures);
  return failures ? 1 : 0;
}

// build_gather against its contract on random sparse rows: each entry names its column in its block's
// list and carries its weight, lists are ascending and padded with their last column; blocks with too
// many columns and weights that are no multiple of 1/32 in (0, 1] are refused.  Exit status 1 on a failure.
#include <cstdio>
#include <random>
#include <vector>

#include "host/octree.hpp"

using namespace dgh;

int main() {
  int failures = 0;
  auto check = [&](bool ok, const char* what) {
    if (!ok && failures++ < 10) std::printf("FAIL %s\n", what);
  };
  std::mt19937 rng(5);
  for (uint32_t nrows : {1u, 31u, 32u, 33u, 1000u})
    for (uint32_t B : {32u, 128u, 256u}) {
      std::vector<uint32_t> ptr(1, 0), col;
      std::vector<float> w;
      for (uint32_t i = 0; i < nrows; ++i) {
        const uint32_t n = rng() % 9;   // empty rows among them
        for (uint32_t k = 0; k < n; ++k) {
          col.push_back((i * 3 + rng() % 700) * 4099u % 100003u);
          w.push_back(float(1 + rng() % 32) / 32.f);
        }
        ptr.push_back(uint32_t(col.size()));
      }
      GatherPlan p;
      check(build_gather(nrows, ptr.data(), col.data(), w.data(), B, p), "accepted");
      for (uint32_t i = 0; i < nrows; ++i)
        for (uint32_t q = ptr[i]; q < ptr[i + 1]; ++q) {
          const uint32_t id = p.ent[q] & GATHER_MAX;
          check(id < p.pitch && p.list[size_t(i / B) * p.pitch + id] == col[q], "column");
          check(float((p.ent[q] >> GATHER_BITS) + 1) / 32.f == w[q], "weight");
        }
      for (size_t i = 1; i < p.list.size(); ++i)
        check(i % p.pitch == 0 || p.list[i] >= p.list[i - 1], "ascending");
      if (w.empty()) continue;
      for (float bad : {0.f, 1.f / 64.f, 33.f / 32.f}) {
        std::vector<float> wb(w);
        wb[rng() % wb.size()] = bad;
        check(!build_gather(nrows, ptr.data(), col.data(), wb.data(), B, p), "weight refused");
      }
    }
  for (uint32_t n : {GATHER_MAX, GATHER_MAX + 1}) {
    std::vector<uint32_t> ptr{0, n}, col(n);
    std::vector<float> w(n, 1.f);
    for (uint32_t i = 0; i < n; ++i) col[i] = n - i;
    GatherPlan p;
    check(build_gather(1, ptr.data(), col.data(), w.data(), 32, p) == (n == GATHER_MAX), "column limit");
  }
  std::printf("%s (%d failures)\n", failures ? "FAILED" : "OK", failures);
  return failures ? 1 : 0;
}

// A few host threads for the planners.
#pragma once

#include <algorithm>
#include <exception>
#include <thread>
#include <vector>

namespace dgh {

// Threads for n pieces of work of which a thread's start is worth `per`.
inline unsigned worker_count(size_t n, size_t per) {
  const size_t most = std::min<size_t>(16, std::max(1u, std::thread::hardware_concurrency()));
  return unsigned(std::min(most, std::max<size_t>(1, n / per)));
}

// Runs f(w) for w = 0 .. nt - 1, the first on the calling thread, and returns when all have ended.  A
// share whose thread cannot be started is run here as well; the first exception (in order of w) is
// thrown again.
template <class F>
void run_workers(unsigned nt, F f) {
  std::vector<std::exception_ptr> err(nt);
  auto share = [&](unsigned w) noexcept {
    try {
      f(w);
    } catch (...) {
      err[w] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  unsigned started = 1;
  try {
    th.reserve(nt);
    for (; started < nt; ++started) th.emplace_back(share, started);
  } catch (...) {   // no thread or no memory for one
  }
  if (nt) share(0);
  for (unsigned w = started; w < nt; ++w) share(w);
  for (std::thread& t : th) t.join();
  for (const std::exception_ptr& e : err)
    if (e) std::rethrow_exception(e);
}

}  // namespace dgh

// Host-side helpers of the library.
#pragma once

#include <algorithm>
#include <cstddef>
#include <thread>
#include <vector>

namespace mose {

// f(first, last) over [0, n) in the host's threads (the plan of a large case: 0.3 us a record).  f does not throw.  Parts
// whose thread cannot be had run on the calling one, so that no exception leaves with threads unjoined, which would end
// the process.
template <class F>
void host_parallel(size_t n, F f) {
  const size_t parts = n < 32768 ? 1 : std::min<size_t>(8, std::max(1u, std::thread::hardware_concurrency()));
  std::vector<std::thread> th;
  th.reserve(parts);
  size_t t = 1;
  try {
    for (; t < parts; ++t) th.emplace_back(f, n * t / parts, n * (t + 1) / parts);
  } catch (...) {
  }
  f((size_t)0, n / parts);
  for (; t < parts; ++t) f(n * t / parts, n * (t + 1) / parts);
  for (auto& q : th) q.join();
}

}  // namespace mose

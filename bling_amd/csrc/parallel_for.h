// Loops over host arrays on several threads.
#pragma once
#include <algorithm>
#include <cstddef>
#include <thread>
#include <vector>

namespace bgpu {

// Runs f(begin, end) over [0, n) in contiguous chunks on up to 16 threads.
template <class F>
void parallel_for(size_t n, F&& f, size_t grain = 32768) {
  const size_t t = std::min<size_t>(16, std::max(1u, std::thread::hardware_concurrency()));
  const size_t k = std::min(t, n / grain);
  if (k <= 1) {
    f((size_t)0, n);
    return;
  }
  std::vector<std::thread> th;
  for (size_t i = 0; i < k; ++i) th.emplace_back([&f, n, k, i] { f(n * i / k, n * (i + 1) / k); });
  for (auto& x : th) x.join();
}

}  // namespace bgpu

// Loops over host arrays on several threads.
#pragma once
#include <algorithm>
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace bgpu {

// Runs f(begin, end) over [0, n) in contiguous chunks on up to 16 threads, or on
// as many as the system grants: what no thread could be started for is done
// here, so that callers behind the C interface see no exception for it.
template <class F>
void parallel_for(size_t n, F&& f, size_t grain = 32768) {
  const size_t t = std::min<size_t>(16, std::max(1u, std::thread::hardware_concurrency()));
  const size_t k = std::min(t, n / grain);
  if (k <= 1) {
    f((size_t)0, n);
    return;
  }
  std::vector<std::thread> th;
  th.reserve(k);
  size_t i = 0;
  try {
    for (; i < k; ++i) th.emplace_back([&f, n, k, i] { f(n * i / k, n * (i + 1) / k); });
  } catch (const std::exception&) {
  }
  if (i < k) f(n * i / k, n);
  for (auto& x : th) x.join();
}

}  // namespace bgpu

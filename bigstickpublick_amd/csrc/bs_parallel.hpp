// body(0) .. body(n - 1) on up to 16 host threads, in any order.  An exception of a body
// ends the others' work early and is thrown on; where no thread can be started, fewer
// (or the caller's alone) do the work.
#pragma once
#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace bs {

template <typename F>
void parallel(int n, F&& body) {
  std::atomic<int> next(0);
  std::exception_ptr thrown;
  std::mutex m;
  auto work = [&]() noexcept {
    try {
      for (int i = next++; i < n; i = next++) body(i);
    } catch (...) {
      next = n;
      std::lock_guard<std::mutex> lock(m);
      if (!thrown) thrown = std::current_exception();
    }
  };
  const int nt = std::min((int)std::min(16u, std::max(1u, std::thread::hardware_concurrency())), n);
  std::vector<std::thread> th;
  th.reserve(16);
  try {
    for (int i = 1; i < nt; i++) th.emplace_back(work);
  } catch (const std::system_error&) {
  }
  work();
  for (auto& q : th) q.join();
  if (thrown) std::rethrow_exception(thrown);
}

}  // namespace bs

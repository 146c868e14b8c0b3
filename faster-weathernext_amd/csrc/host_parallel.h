// Dynamic parallel loop of the host pipeline.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace fwn {

inline int worker_count() {
  unsigned hw = std::thread::hardware_concurrency();
  if (hw == 0) hw = 4;
  return (int)std::min<unsigned>(hw, 16);
}

// Runs fn(begin, end) over [0, n) split into chunks handed out dynamically to the workers. An
// exception in a worker ends the loop and is thrown again in the caller.
template <typename Fn>
void parallel_for(int64_t n, int64_t grain, Fn fn) {
  int workers = (int)std::min<int64_t>(worker_count(), (n + grain - 1) / grain);
  if (workers <= 1) {
    fn((int64_t)0, n);
    return;
  }
  std::atomic<int64_t> next(0);
  std::exception_ptr error;
  std::mutex error_mu;
  auto work = [&]() {
    try {
      for (;;) {
        int64_t b = next.fetch_add(grain);
        if (b >= n) break;
        fn(b, std::min(n, b + grain));
      }
    } catch (...) {
      next = n;
      std::lock_guard<std::mutex> lock(error_mu);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  try {
    for (int w = 1; w < workers; ++w) pool.emplace_back(work);
  } catch (...) {
    // Fewer threads than asked for: the ones that started and this one do the work.
  }
  work();
  for (auto& t : pool) t.join();
  if (error) std::rethrow_exception(error);
}

}  // namespace fwn

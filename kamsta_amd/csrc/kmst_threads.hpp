// kmst_threads.hpp -- work on host data by several threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace kmst {

// f(t) for t < `threads` at most, t = 0 on the caller's thread; the first
// failure is thrown once all have ended.  Where the system has no thread or no
// memory for one, only the lower t run: f draws its share of the work from a
// counter that all share, and does all of it if it runs alone.
template <typename F>
void on_threads(unsigned threads, F&& f) {
  std::mutex mu;
  std::exception_ptr failure;
  auto run = [&](unsigned t) {
    try {
      f(t);
    } catch (...) {
      std::lock_guard<std::mutex> lk(mu);
      if (!failure) failure = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  try {
    th.reserve(threads ? threads - 1 : 0);  // no growth beside running threads
    for (unsigned t = 1; t < threads; ++t) th.emplace_back(run, t);
  } catch (...) {
  }
  run(0);
  for (auto& x : th) x.join();
  if (failure) std::rethrow_exception(failure);
}

// f(first, last) over the blocks of `block` items of [0, n), drawn in turn.
template <typename F>
void for_blocks(unsigned threads, std::uint64_t n, std::uint64_t block, F&& f) {
  std::atomic<std::uint64_t> next{0};
  on_threads(threads, [&](unsigned) {
    for (std::uint64_t at; (at = next.fetch_add(block)) < n;) f(at, std::min(n, at + block));
  });
}

}  // namespace kmst

// Host work shared by a few threads.
#pragma once
#include <algorithm>
#include <atomic>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

// f(g, scratch) for every g < n, by up to `threads` threads, each with a Scratch of its own;
// std::bad_alloc where one ran out of memory.
// Nothing leaves with a thread running: one that cannot be started, for want of threads or
// of memory, leaves its share to those there are.
template <typename Scratch, typename F>
void parallel_for(int n, int threads, const F& f) {
  std::atomic<int> next(0);
  std::atomic<bool> nomem(false);
  auto work = [&] {
    try {
      Scratch scratch{};
      for (int g; (g = next.fetch_add(1)) < n;) f(g, scratch);
    } catch (const std::bad_alloc&) {      // nothing may leave a thread
      nomem = true;
    }
  };
  const int nt = std::max(1, std::min({threads, (int)std::thread::hardware_concurrency(), n}));
  std::vector<std::thread> pool;
  pool.reserve(nt);
  try {
    for (int k = 1; k < nt; ++k) pool.emplace_back(work);
  } catch (const std::system_error&) {
  } catch (const std::bad_alloc&) {
  }
  work();
  for (std::thread& th : pool) th.join();
  if (nomem) throw std::bad_alloc();
}

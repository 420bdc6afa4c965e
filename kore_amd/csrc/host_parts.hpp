// Work of an entry point split over host threads.
#pragma once
#include <algorithm>
#include <exception>
#include <thread>
#include <vector>

// f(0) .. f(n - 1), f(0) on this thread and the others on threads of their own; parts
// whose thread cannot be started (the process or user is at its limit) run here too, so
// that no exception leaves an entry point for want of a thread.
template <class F> void run_parts(int n, F&& f) {
  std::vector<std::thread> pool;
  int started = 1;
  try {
    pool.reserve((size_t)std::max(0, n - 1));
    for (; started < n; ++started) pool.emplace_back([&f, t = started] { f(t); });
  } catch (const std::exception&) {        // std::system_error, std::bad_alloc
  }
  for (int t = started; t < n; ++t) f(t);
  f(0);
  for (std::thread& x : pool) x.join();
}

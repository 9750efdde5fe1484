// Helper threads of a host-side pipeline behind a C entry point, where an exception must not pass.
#pragma once
#include <sched.h>
#include <thread>
#include <vector>

// How many helpers beside the caller are worth starting: at most `most`, and no more than the calling thread may use cores beside its own.
inline int helper_count(int most) {
  cpu_set_t set; CPU_ZERO(&set);
  const int cores = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 0;          // (0: not to be had, or more cores than the set holds)
  return most < 0 ? 0 : (cores > 0 && most > cores - 1 ? cores - 1 : most);
}
// Starts f(1) .. f(n) on threads of their own; a system that refuses one (a process limit, no memory) leaves the caller
// with those that were started -- th.size() of them, to be joined as usual.  Noexcept: f's copies must not throw.
template <class F> void start_helpers(std::vector<std::thread>& th, int n, const F& f) noexcept {
  try {
    th.reserve((size_t)(n > 0 ? n : 0));
    for (int w = 1; w <= n; ++w) th.emplace_back([&f, w] { f(w); });
  } catch (...) {}
}

// pdt_pool.hpp -- host threads of the concurrent solves.
#pragma once

#include <algorithm>
#include <system_error>
#include <thread>
#include <vector>

namespace pdt {

// Runs work() on the calling thread and on up to count - 1 more, and returns
// when all have.  work must not throw and must leave nothing to a given number
// of callers: a thread that cannot be started (the limit of the process, no
// memory for its stack) is done without.
template <class F>
void run_workers(int count, F&& work) {
  std::vector<std::thread> pool;
  pool.reserve(size_t(std::max(count, 1)));
  try {
    while (int(pool.size()) + 1 < count) pool.emplace_back([&work] { work(); });
  } catch (const std::system_error&) {
  }
  work();
  for (auto& t : pool) t.join();
}

}  // namespace pdt

// Threads that cannot be started: the address space is limited to what the
// process has and a few thread stacks, then 64 workers take 1000 items.
#include <sys/resource.h>

#include <atomic>
#include <cstdio>
#include <fstream>
#include <string>

#include "pdt_pool.hpp"

int main() {
  std::ifstream in("/proc/self/statm");
  long pages = 0;
  in >> pages;
  const rlim_t bytes = rlim_t(pages) * 4096 + (rlim_t(64) << 20);
  const rlimit lim{bytes, bytes};
  if (setrlimit(RLIMIT_AS, &lim) != 0) return 2;
  std::atomic<int> next{0}, done{0}, workers{0};
  pdt::run_workers(64, [&] {
    workers++;
    while (next++ < 1000) done++;
  });
  std::printf("%d items, %d workers\n", done.load(), workers.load());
  return done == 1000 && workers < 64 ? 0 : 1;
}

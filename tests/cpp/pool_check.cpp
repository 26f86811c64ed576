// host_parallel (cf_host.cpp): every item is visited exactly once, whoever calls it: from
// several threads at once, with and without a holder, across restarts of the pool, and in a
// forked child.  Exits 0 when all hold.
#include <sys/wait.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "../../cellflow_amd/csrc/cf_host.h"

static bool once(size_t n, size_t grain) {
  std::vector<std::atomic<int>> seen(n);
  std::atomic<bool> big{false};
  cf::host_parallel(n, grain, [&](size_t i0, size_t i1) {
    if (i1 - i0 > std::max<size_t>(grain, 1) && i1 - i0 != n) big = true;
    for (size_t i = i0; i < i1; ++i) seen[i]++;
  });
  for (size_t i = 0; i < n; ++i)
    if (seen[i] != 1) return false;
  return !big;
}

static bool several(int rounds) {
  std::atomic<bool> ok{true};
  std::vector<std::thread> t;
  for (int k = 0; k < 4; ++k)
    t.emplace_back([&, k] {
      for (int r = 0; r < rounds; ++r)
        if (!once(1000 + 37 * k + r, 16)) ok = false;
    });
  for (auto& x : t) x.join();
  return ok;
}

int main() {
  if (!once(0, 8) || !once(1, 8) || !once(5000, 8)) return 1;  // no holder
  for (int cycle = 0; cycle < 20; ++cycle) {
    cf::host_pool_hold();
    cf::host_pool_hold();
    for (size_t n : {0u, 1u, 23u, 24u, 25u, 1000u, 4097u})
      if (!once(n, 8)) return 2;
    if (!once(100, 0)) return 3;
    if (!several(50)) return 4;
    cf::host_pool_drop();
    if (!once(4097, 8)) return 5;
    cf::host_pool_drop();
    if (!once(4097, 8)) return 6;
  }
  cf::host_pool_hold();
  if (!once(4097, 8)) return 7;
  const pid_t child = fork();
  if (child == 0) {
    const bool ok = once(4097, 8);
    cf::host_pool_drop();
    _exit(ok ? 0 : 1);
  }
  int st = 0;
  if (waitpid(child, &st, 0) != child || !WIFEXITED(st) || WEXITSTATUS(st) != 0) return 8;
  if (!once(4097, 8)) return 9;
  cf::host_pool_drop();
  std::puts("pool ok");
  return 0;
}

// When host_parallel's threads (cf_host.cpp) exist: never for small jobs, kHostHelpers from the
// first larger one on until the last holder is gone.  Exits 0 when all hold.
#include <dirent.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <thread>

#include "../../cellflow_amd/csrc/cf_host.h"

// Threads of this process.
static int threads() {
  DIR* d = opendir("/proc/self/task");
  int n = 0;
  while (const dirent* e = readdir(d)) n += e->d_name[0] != '.';
  closedir(d);
  return n;
}

// Whether `n` more threads exist than the process began with (an ended thread's entry may
// outlive its join for a moment).
static int began = 0;
static bool extra(int n) {
  for (int k = 0; k < 1000 && threads() != began + n; ++k) usleep(1000);
  return threads() == began + n;
}

// A job of `items` items in ranges of 100; false: not every item was visited.
static bool job(size_t items) {
  std::atomic<size_t> done{0};
  cf::host_parallel(items, 100, [&](size_t i0, size_t i1) { done += i1 - i0; });
  return done == items;
}

int main() {
  std::thread([] {}).join();  // a sanitizer's own thread comes with the first
  usleep(10000);
  began = threads();
  const size_t small = cf::kHostAlone * 100;
  for (int cycle = 0; cycle < 4; ++cycle) {
    if (!job(100000)) return 1;  // no holder
    cf::host_pool_hold();
    for (int k = 0; k < 1000; ++k)
      if (!job(small)) return 2;
    if (!extra(0)) return 3;
    for (int k = 0; k < (cycle == 0 ? 1 : 20); ++k) {
      if (!job(k == 0 ? small + 1 : 100000)) return 4;
      if (cycle < 2 && !extra(cf::kHostHelpers)) return 5;  // later: without a pause
    }
    cf::host_pool_hold();  // they belong to the process, not to one holder
    cf::host_pool_drop();
    if (cycle < 3 && !extra(cf::kHostHelpers)) return 6;
    if (cycle % 2) {
      cf::host_pool_drop();
    } else {  // a holder that begins while the last one's threads end has its own
      cf::HostPool* ending = cf::host_pool_leave();
      cf::host_pool_hold();
      if (!ending || !job(100000)) return 7;
      cf::host_pool_end(ending);
      if (!extra(cf::kHostHelpers)) return 8;
      if (cf::HostPool* last = cf::host_pool_leave()) cf::host_pool_end(last);
    }
    if (!extra(0)) return 9;
    if (!job(100000) || !extra(0)) return 10;
  }
  std::puts("start ok");
  return 0;
}

// Host-only entry points and helpers of the C ABI: the error string, tuning validation and
// the tuning-cache file calls.  No device code.

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "cf_host.h"
#include "cf_tune_cache.h"

namespace cf {

std::string& error_text() {
  static thread_local std::string text;
  return text;
}

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  error_text() = buf;
  return code;
}

struct HostPool {
  std::mutex mu;
  std::condition_variable wake, done;
  std::thread first;
  std::vector<std::thread> rest;  // the first thread's until it ends
  const std::function<void(size_t, size_t)>* fn = nullptr;  // the job, null between jobs
  size_t n = 0, grain = 0;
  std::atomic<size_t> next{0};
  unsigned long long job = 0;
  int active = 0;
  bool stop = false;

  void take(const std::function<void(size_t, size_t)>& f, size_t count, size_t step) {
    for (size_t i = next.fetch_add(step); i < count; i = next.fetch_add(step))
      f(i, std::min(count, i + step));
  }

  // The first thread starts the others, so that the job it was started for waits for one.
  void lead() {
    try {
      while ((int)rest.size() + 1 < kHostHelpers) rest.emplace_back([this] { work(); });
    } catch (...) {  // as many as the system gives
    }
    work();
  }

  void work() {
    unsigned long long seen = 0;
    std::unique_lock<std::mutex> l(mu);
    while (true) {
      wake.wait(l, [&] { return stop || job != seen; });
      if (stop) return;
      seen = job;
      if (!fn) continue;  // the job ended before this thread woke
      const auto* f = fn;
      const size_t count = n, step = grain;
      ++active;
      l.unlock();
      take(*f, count, step);
      l.lock();
      if (--active == 0) done.notify_all();
    }
  }
};

namespace {

std::mutex g_pool_mu;  // guards the three below
std::mutex g_run_mu;   // one job at a time
HostPool* g_pool = nullptr;
int g_pool_users = 0;
std::atomic<pid_t> g_pool_pid{0};  // the process the threads live in

}  // namespace

void host_pool_hold() {
  std::lock_guard<std::mutex> l(g_pool_mu);
  ++g_pool_users;
}

HostPool* host_pool_leave() {
  const pid_t owner = g_pool_pid.load();
  if (owner != 0 && owner != getpid()) return nullptr;  // a forked child has none of the threads
  HostPool* gone = nullptr;
  {
    std::lock_guard<std::mutex> l(g_pool_mu);
    if (--g_pool_users == 0) {
      gone = g_pool;
      g_pool = nullptr;
      g_pool_pid = 0;
    }
  }
  if (!gone) return nullptr;
  {
    std::lock_guard<std::mutex> l(gone->mu);
    gone->stop = true;
  }
  gone->wake.notify_all();
  return gone;
}

void host_pool_end(HostPool* gone) {
  if (!gone) return;
  if (gone->first.joinable()) gone->first.join();
  for (std::thread& t : gone->rest) t.join();
  delete gone;
}

void host_pool_drop() { host_pool_end(host_pool_leave()); }

void host_parallel(size_t n, size_t grain, const std::function<void(size_t, size_t)>& fn) {
  grain = std::max<size_t>(grain, 1);
  const pid_t owner = g_pool_pid.load();
  std::unique_lock<std::mutex> run(g_run_mu, std::defer_lock);
  if (n <= kHostAlone * grain || (owner != 0 && owner != getpid()) || !run.try_lock()) {
    if (n) fn(0, n);
    return;
  }
  HostPool* p = nullptr;
  {
    std::unique_lock<std::mutex> l(g_pool_mu, std::try_to_lock);
    if (l && g_pool_users > 0) {
      if (!g_pool) {
        g_pool = new (std::nothrow) HostPool;
        if (g_pool) {
          g_pool_pid = getpid();
          try {
            g_pool->first = std::thread([q = g_pool] { q->lead(); });
          } catch (...) {  // none to be had: the callers do everything
          }
        }
      }
      p = g_pool;
    }
  }
  // the pool outlives this call: the caller's engine holds it
  if (!p) {
    fn(0, n);
    return;
  }
  {
    std::lock_guard<std::mutex> l(p->mu);
    p->fn = &fn;
    p->n = n;
    p->grain = grain;
    p->next = 0;
    ++p->job;
  }
  p->wake.notify_all();
  p->take(fn, n, grain);
  std::unique_lock<std::mutex> l(p->mu);
  p->fn = nullptr;  // a helper that wakes from here on skips the job
  p->done.wait(l, [&] { return p->active == 0; });
}

int check_tuning(const cf_tuning* t) {
  if (!t) return fail(CF_ERR_ARG, "tuning is null");
  if (t->cell_divisor != 1 && t->cell_divisor != 2)
    return fail(CF_ERR_ARG, "cell_divisor must be 1 or 2");
  if (t->block_size != 64 && t->block_size != 128 && t->block_size != 256)
    return fail(CF_ERR_ARG, "block_size must be 64, 128 or 256");
  if (t->force_variant < 0 || t->force_variant > 4)
    return fail(CF_ERR_ARG, "force_variant must be 0, 1, 2, 3 or 4");
  if (t->force_variant == 4 && t->lanes_per_particle != 8 && t->lanes_per_particle != 16)
    return fail(CF_ERR_ARG, "force_variant 4 needs lanes_per_particle 8 or 16");
  if (t->lanes_per_particle != 4 && t->lanes_per_particle != 8 && t->lanes_per_particle != 16 &&
      t->lanes_per_particle != 32)
    return fail(CF_ERR_ARG, "lanes_per_particle must be 4, 8, 16 or 32");
  if (t->force_variant == 3 && t->lanes_per_particle < 4 * t->cell_divisor)
    return fail(CF_ERR_ARG, "force_variant 3 needs lanes_per_particle >= 8 with cell_divisor 2");
  if (t->steps_per_graph < 1) return fail(CF_ERR_ARG, "steps_per_graph must be >= 1");
  if (t->sort_variant != 0 && t->sort_variant != 1)
    return fail(CF_ERR_ARG, "sort_variant must be 0 or 1");
  return CF_OK;
}

}  // namespace cf

extern "C" {

const char* cf_last_error_string(void) { return cf::error_text().c_str(); }

int cf_tuning_cache_lookup(const char* cache_path, const char* key, cf_tuning* tuning,
                           double* us_per_step, int* found) {
  if (!cache_path || !key || !tuning || !found) return cf::fail(CF_ERR_ARG, "null argument");
  *found = 0;
  std::map<std::string, cf::tunecache::Entry> ents;
  std::string why;
  const int st = cf::tunecache::read_file(cache_path, ents, why);
  if (st == cf::tunecache::kBad)
    return cf::fail(CF_ERR_ARG, "tuning cache %s: %s", cache_path, why.c_str());
  auto it = ents.find(key);
  if (it == ents.end() || !cf::tunecache::valid(it->second.tun)) return CF_OK;
  *tuning = it->second.tun;
  if (us_per_step) *us_per_step = it->second.us;
  *found = 1;
  return CF_OK;
}

int cf_tuning_cache_store(const char* cache_path, const char* key, const cf_tuning* tuning,
                          double us_per_step) {
  if (!cache_path || !key) return cf::fail(CF_ERR_ARG, "null argument");
  const int rc = cf::check_tuning(tuning);
  if (rc != CF_OK) return rc;
  if (!std::isfinite(us_per_step)) return cf::fail(CF_ERR_ARG, "us_per_step must be finite");
  std::map<std::string, cf::tunecache::Entry> ents;
  std::string why;
  const int st = cf::tunecache::read_file(cache_path, ents, why);
  if (st == cf::tunecache::kBad)
    return cf::fail(CF_ERR_ARG, "tuning cache %s: %s", cache_path, why.c_str());
  ents[key] = cf::tunecache::Entry{*tuning, us_per_step};
  if (!cf::tunecache::write_file(cache_path, ents, why))
    return cf::fail(CF_ERR_ARG, "cannot write tuning cache %s: %s", cache_path, why.c_str());
  return CF_OK;
}

}  // extern "C"

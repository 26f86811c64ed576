// Host-only helpers shared by the engine (cf_engine.hip) and the host-only sources
// (cf_preset.cpp, cf_host.cpp).  No HIP headers: the host-only sources also build with a
// plain C++ compiler (the sanitizer build of the tests).
#pragma once

#include <cstddef>
#include <functional>
#include <string>

#include "../../include/cellflow.h"

namespace cf {

// Records the message of a failing call (read back by cf_last_error_string) and returns
// `code`.
int fail(int code, const char* fmt, ...);
// The calling thread's last error message.
std::string& error_text();
// CF_OK when every field of `t` holds an allowed value, else CF_ERR_ARG with the reason.
int check_tuning(const cf_tuning* t);

// A few helper threads for the host side of large loads and readbacks: one core copies about
// 10 GB/s between pinned and pageable memory, a fifth of what the DMA beside it moves (100k
// particles' records, 4.4 MB: 0.45 ms of copying against 0.09).  The process has at most one
// pool of kHostHelpers threads; it starts with the first large copy while an engine lives
// and ends with the last engine.
constexpr int kHostHelpers = 3;
void host_pool_hold();  // an engine begins to live
void host_pool_drop();  // and ends: the last one joins the threads
// fn(begin, end) over disjoint ranges of at most `grain` items that cover [0, n), by the
// caller and the helpers; returns when all are done.  Up to three ranges, another thread's call in progress, a
// forked child, or no engine: the caller does everything itself.  fn must not throw.
void host_parallel(size_t n, size_t grain, const std::function<void(size_t, size_t)>& fn);

}  // namespace cf

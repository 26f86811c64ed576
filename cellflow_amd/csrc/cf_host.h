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

// A few helper threads for the host side of large loads and readbacks, whose copies between
// pinned and pageable memory take longer than the DMA beside them.  The process has at most one
// pool of kHostHelpers threads while an engine lives; it ends with the last engine.
//
// Measured as whole readbacks of particle records, repeated, by one thread and by four (ranges
// of 128 KiB): 0.40 MB 42 -> 47 us, 0.53 MB 46 -> 50, 0.79 MB 56 -> 59, 1.1 MB 82 -> 67,
// 2.2 MB 136 -> 108, 4.4 MB 245 -> 162, 22 MB 1150 -> 653; and of the copies alone into memory
// that was never touched: 0.4 MB 60 -> 40, 1.0 MB 158 -> 93, 4.4 MB 962 -> 398.  Hence kHostAlone:
// up to 768 KiB waking the threads costs a repeated copy more than they take over.
// The threads begin with the first larger job, which starts one that starts the others, and end
// while the last engine frees its memory.  Started by the job and joined after the frees, they
// made a program that opens an engine, loads, steps once, reads and ends slower (1.1 MB of
// records: 976 us, 876 without threads; now 994 against 1021 and 1007 on another machine; 0.40 MB:
// 795, 769 without, 682 now).  Started only once jobs add up to 3 MiB, they came late for the
// first pass over new buffers (7.8 MB of vertices and edges: 2960 -> 3150 us, 4700 without).
constexpr int kHostHelpers = 3;
constexpr size_t kHostAlone = 6;  // ranges that the caller does by itself
struct HostPool;
void host_pool_hold();  // an engine begins to live
// ... and ends: the last one is given the pool, whose threads it has told to end, and waits
// for them with host_pool_end (null: nothing to wait for) when its own work is done.
HostPool* host_pool_leave();
void host_pool_end(HostPool* gone);
void host_pool_drop();  // both at once
// fn(begin, end) over disjoint ranges of at most `grain` items that cover [0, n), by the
// caller and the helpers; returns when all are done.  Up to kHostAlone ranges, another thread's
// call in progress, a forked child, or no engine: the caller does everything itself.  fn must
// not throw.
void host_parallel(size_t n, size_t grain, const std::function<void(size_t, size_t)>& fn);

}  // namespace cf

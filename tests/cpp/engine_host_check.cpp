// The engine's host side against a HIP runtime that lives in this program: device memory is
// host memory, a kernel launch is a line of the log, and any allocation can be made to fail.
// The definitions here come before the real runtime's in symbol order, so libcellflow.so binds
// to them; nothing needs a GPU.  Each case checks which calls the engine makes, and that none
// of them touches memory that was never allocated or was freed.
//
//   engine_host_check CASE   exits 0 when the case holds
#include <hip/hip_runtime_api.h>

#include <sys/resource.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "cellflow.h"

// ---- the runtime -----------------------------------------------------------------------

namespace {

struct Runtime {
  std::map<const void*, std::string> kernels;   // host function -> device name
  std::map<const char*, size_t> mem;            // live allocations
  std::vector<std::string> log;
  hipError_t last = hipSuccess;
  int device = 0;                               // the current one, of two
  // the countdowns reach a failure at 0; negative: never
  int fail_malloc = -1, fail_copy = -1;
  bool fail_info = false;                       // hipMemGetInfo fails
  size_t host_limit = ~size_t(0);               // larger pinned allocations fail
  uint32_t edges = 0;                           // the graph's size in the status words read back
  dim3 grid, block;
  size_t shm = 0;
  hipStream_t stream = nullptr;
};

Runtime& rt() {
  static Runtime* r = new Runtime;  // outlives the library's own destructors
  return *r;
}

hipError_t result(hipError_t e) {
  if (e != hipSuccess) rt().last = e;
  return e;
}

bool due(int& countdown) { return countdown >= 0 && countdown-- == 0; }

[[noreturn]] void die(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  std::vfprintf(stderr, fmt, ap);
  va_end(ap);
  std::fputc('\n', stderr);
  std::_Exit(1);
}

// Whether [p, p + n) lies in one live allocation.
bool live(const void* p, size_t n) {
  const char* c = (const char*)p;
  auto it = rt().mem.upper_bound(c);
  if (it == rt().mem.begin()) return false;
  --it;
  return c + n <= it->first + it->second;
}

hipError_t allocate(void** p, size_t n) {
  char* c = (char*)std::calloc(1, n);
  rt().mem[c] = n;
  *p = c;
  return hipSuccess;
}

hipError_t release(void* p) {
  if (!rt().mem.erase((const char*)p)) die("free of %p, which is not allocated", p);
  std::free(p);
  return hipSuccess;
}

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  rt().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shm, hipStream_t st) {
  rt().grid = grid;
  rt().block = block;
  rt().shm = shm;
  rt().stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shm, hipStream_t* st) {
  *grid = rt().grid;
  *block = rt().block;
  *shm = rt().shm;
  *st = rt().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
  auto it = rt().kernels.find(f);
  if (it == rt().kernels.end()) die("launch of an unknown kernel");
  rt().log.push_back(it->second);
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = rt().device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  rt().device = d;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = rt().last;
  rt().last = hipSuccess;
  return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return allocate(p, 64); }
hipError_t hipMemGetInfo(size_t* avail, size_t* total) {
  if (rt().fail_info) return result(hipErrorInvalidValue);
  *avail = *total = size_t(256) << 30;
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  rt().log.push_back("malloc");
  if (due(rt().fail_malloc)) return result(hipErrorOutOfMemory);
  return allocate(p, n);
}
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (n > rt().host_limit) return result(hipErrorOutOfMemory);
  return allocate(p, n);
}
hipError_t hipHostFree(void* p) { return release(p); }

hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  if (!live(p, n)) die("memset of %zu bytes at %p", n, p);
  std::memset(p, v, n);
  rt().log.push_back("memset");
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
  if (kind != hipMemcpyDeviceToHost && !live(d, n)) die("copy of %zu bytes to %p", n, d);
  if (kind != hipMemcpyHostToDevice && !live(s, n)) die("copy of %zu bytes from %p", n, s);
  if (due(rt().fail_copy)) return result(hipErrorUnknown);
  std::memcpy(d, s, n);
  if (kind == hipMemcpyDeviceToHost && n == 4 * sizeof(uint32_t)) ((uint32_t*)d)[1] = rt().edges;
  rt().log.push_back("copy");
  return hipSuccess;
}

// a stream and an event are known by the device they were made on
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t) new int(rt().device);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete (int*)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  rt().log.push_back("sync");
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t) new int(rt().device);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return result(*(int*)e == *(int*)s ? hipSuccess : hipErrorInvalidHandle);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (int*)e;
  return hipSuccess;
}

}  // extern "C"

// ---- the cases -------------------------------------------------------------------------

namespace {

#define HOLDS(x)                                                        \
  do {                                                                  \
    if (!(x)) die("line %d: %s does not hold", __LINE__, #x);           \
  } while (0)
#define OK(x)                                                           \
  do {                                                                  \
    const int rc_ = (x);                                                \
    if (rc_ != CF_OK) die("line %d: %s: %s", __LINE__, #x, cf_last_error_string()); \
  } while (0)

cf_params params(float radius, float side) {
  cf_params p{};
  p.radius = radius;
  p.delta_t = 0.01f;
  p.friction = 0.9f;
  p.repulsion = p.attraction = p.k = 1.0f;
  p.canvas_width = p.canvas_height = p.canvas_depth = side;
  p.num_particle_types = 2;
  p.force_multiplier = 1.0f;
  p.max_expected_neighbors = 100;
  return p;
}

int logged(const char* what) {
  int k = 0;
  for (const std::string& s : rt().log) k += s.find(what) != std::string::npos;
  return k;
}

struct Sim {
  cf_sim* h = nullptr;
  int n;
  explicit Sim(int count) : n(count) { OK(cf_create(count, 2, &h)); }
  ~Sim() { OK(cf_destroy(h)); }
};

// Every allocation of a call that needs larger buffers fails once, in turn: the call reports
// it, and the next calls, at the old sizes and at the new, allocate what the failed one gave
// up and sort the state again before they walk its cells.
void grow_cells() {
  const cf_params coarse = params(0.2f, 2.0f), fine = params(0.05f, 2.0f);
  const cf_edge_opts few{0.02f, 4}, many{0.02f, 16};
  for (const bool edges : {false, true}) {
    for (const bool back : {false, true}) {
      int failures = 0;
      for (int k = 0;; ++k) {
        Sim s(20000);
        const cf_params& next = edges ? coarse : fine;
        OK(cf_simulate(s.h, &coarse, 2, edges ? &few : nullptr));
        rt().fail_malloc = k;
        const int rc = cf_simulate(s.h, &next, 2, edges ? &many : nullptr);
        const bool failed = rt().fail_malloc < 0;
        rt().fail_malloc = -1;
        HOLDS(failed == (rc == CF_ERR_DEVICE));
        if (!failed) break;
        ++failures;
        double hist[8];
        rt().log.clear();
        if (!edges) HOLDS(cf_pair_histogram_noalloc(s.h, 8, 0.05f, hist) == CF_ERR_STATE);
        HOLDS(logged("k_") == 0);
        OK(cf_simulate(s.h, back ? &coarse : &next, 2,
                       !edges ? nullptr : back ? &few : &many));
        HOLDS(logged("malloc") > 0);
        if (!edges) HOLDS(logged("k_bin") == 1);
        rt().log.clear();
        OK(cf_simulate(s.h, back ? &coarse : &next, 2,
                       !edges ? nullptr : back ? &few : &many));
        HOLDS(logged("malloc") == 0 && logged("k_bin") == 0);
      }
      HOLDS(failures >= (edges ? 5 : 6));
    }
  }
}

// The calls that change a whole state have nothing outstanding when they return.
void changes_wait() {
  const cf_params p = params(0.1f, 2.0f);
  const float canvas[3] = {2.0f, 2.0f, 2.0f};
  Sim s(5000);
  OK(cf_simulate(s.h, &p, 3, nullptr));
  for (int k = 0; k < 2; ++k) {  // with and without new descriptors before
    rt().log.clear();
    OK(cf_move_universe(s.h, 0.1f, 0.2f, 0.0f, canvas));
    HOLDS(logged("k_move") == 1 && rt().log.back() == "sync");
    rt().log.clear();
    OK(cf_init_particles(s.h, 3, canvas, 1.0f));
    HOLDS(logged("k_init") == 1 && rt().log.back() == "sync");
  }
}

// Where the system pins little memory, loads and readbacks do without the staging buffer.
void pins_little() {
  Sim s(60000);  // 2.6 MB of records: two slices of the staged path
  std::vector<cf_particle> in(s.n), out(s.n);
  std::vector<int32_t> counts(s.n);
  for (int round = 0; round < 4; ++round) {
    rt().host_limit = round % 2 ? ~size_t(0) : size_t(1) << 16;
    for (int i = 0; i < s.n; ++i) {
      in[i].pos[0] = (float)(i + round);
      in[i].ptype = (uint32_t)(i & 1);
    }
    OK(cf_set_particles(s.h, in.data(), s.n));
    // nothing ran between, so what is read back is what the load left in the device buffer
    OK(cf_get_particles(s.h, out.data(), s.n));
    HOLDS(std::memcmp(in.data(), out.data(), in.size() * sizeof(cf_particle)) == 0);
    OK(cf_get_neighbor_counts(s.h, counts.data(), s.n));
    HOLDS(std::memcmp(in.data(), counts.data(), counts.size() * sizeof(int32_t)) == 0);
    in[s.n - 1].ptype = 2;
    HOLDS(cf_set_particles(s.h, in.data(), s.n) == CF_ERR_ARG);
    HOLDS(hipGetLastError() == hipSuccess);
  }
}

// Colours are uploaded when they change, and again after an upload that failed.
void colours() {
  const cf_params p = params(0.1f, 2.0f);
  cf_color c[2] = {{1, 0, 0}, {0, 1, 0}};
  Sim s(2000);
  OK(cf_simulate(s.h, &p, 1, nullptr));
  rt().edges = 3;
  OK(cf_build_edges(s.h, 0.05f, 4));
  std::vector<float> out(12 * 3);
  long long count = 0;
  auto draw = [&] {
    rt().log.clear();
    return cf_get_line_vertices(s.h, c, 2, out.data(), (long long)out.size(), &count);
  };
  for (int k = 0; k < 2; ++k) {
    OK(draw());
    HOLDS(count == 6 && logged("copy") == 2);  // the colours up, the vertices down
    OK(draw());
    HOLDS(logged("copy") == 1);
    c[0].g = 0.5f + k;
    rt().fail_copy = 0;
    HOLDS(draw() == CF_ERR_DEVICE);
  }
  OK(draw());
  HOLDS(logged("copy") == 2);
}

// An engine of one device read back by a thread whose current device is another.
void other_device() {
  OK(hipSetDevice(1));
  Sim s(60000);  // two slices
  std::vector<cf_particle> in(s.n), out(s.n);
  for (int i = 0; i < s.n; ++i) in[i].pos[0] = (float)i;
  OK(cf_set_particles(s.h, in.data(), s.n));
  OK(hipSetDevice(0));
  for (int k = 0; k < 2; ++k) {
    OK(cf_get_particles(s.h, out.data(), s.n));
    HOLDS(std::memcmp(in.data(), out.data(), in.size() * sizeof(cf_particle)) == 0);
    HOLDS(rt().device == 0);
  }
}

// A gradient of more steps than could ever all be kept costs the host no memory to find out
// (its checkpoints fit), and a runtime that cannot tell the free memory fails no call.
void long_rollout() {
  cf_params p = params(0.1f, 2.0f);
  double target[4] = {1, 1, 1, 1}, loss = 0, table[4], ratio = 0;
  const rlimit limit{size_t(8) << 30, size_t(8) << 30};
  HOLDS(setrlimit(RLIMIT_AS, &limit) == 0);
  for (const int steps : {1000000000, 100000000}) {
    Sim s(64);
    OK(cf_simulate(s.h, &p, 1, nullptr));
    rt().fail_malloc = 0;  // before a step is run
    HOLDS(cf_rollout_grad(s.h, &p, steps, 1000, 4, 0.1f, target, &loss, nullptr, table, &ratio) ==
          CF_ERR_DEVICE);
    HOLDS(rt().fail_malloc < 0);
  }
  Sim s(64);
  rt().fail_info = true;
  OK(cf_rollout_grad(s.h, &p, 20, 5, 4, 0.1f, target, &loss, nullptr, table, &ratio));
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, std::function<void()>> cases = {
      {"grow_cells", grow_cells},
      {"changes_wait", changes_wait},
      {"pins_little", pins_little},
      {"colours", colours},
      {"other_device", other_device},
      {"long_rollout", long_rollout},
  };
  const auto it = argc == 2 ? cases.find(argv[1]) : cases.end();
  if (it == cases.end()) die("usage: engine_host_check CASE");
  it->second();
  std::printf("%s ok\n", argv[1]);
  return 0;
}

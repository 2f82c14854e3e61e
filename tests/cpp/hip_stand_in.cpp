// A stand-in for the HIP runtime, so that the library's host code can be run
// and its decisions seen without a device: which kernels are launched, what is
// allocated, what happens when an allocation fails.  Device memory is zeroed
// host memory, kernels do nothing but are counted, copies are carried out
// (large ones left out), and time passes only in launches.
//
// Loaded before libqesmc under the runtime's own soname (tests/test_host_runs.py).
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>

namespace {

constexpr size_t kLargest = (size_t)64 << 20;  // copies and fills beyond this are left out
constexpr int kNames = 1024, kLog = 1 << 20, kBlocks = 16384;

struct Name {
  const void *host;
  const char *name;
};
Name g_names[kNames];
int g_nnames = 0;
struct Launch {
  int name;
  unsigned grid;
};
Launch g_log[kLog];
int g_nlog = 0;
struct Block {
  char *p;
  size_t bytes;
  bool device;
};
Block g_blocks[kBlocks];
std::recursive_mutex g_mu;

long long g_fail_at = 0, g_fail_above = 0, g_fail_new = 0;  // 0: never
long long g_device_allocs = 0, g_host_allocs = 0, g_live = 0, g_host_live = 0;
std::atomic<long long> g_news{0};
thread_local bool g_count_news = false;
std::atomic<long long> g_syncs{0}, g_copies{0};
long long g_graph_launches = 0;
bool g_capturing = false;
double g_clock = 0.0;
const char *g_slow = nullptr;
double g_slow_cost = 1.0;

struct Event {
  double at;
};

thread_local struct {
  unsigned g[3], b[3];
  size_t shm;
  void *stream;
} g_config;

int allocate(void **p, size_t bytes, bool device)
{
  std::lock_guard<std::recursive_mutex> lock(g_mu);
  ++(device ? g_device_allocs : g_host_allocs);
  *p = nullptr;
  if (device && g_fail_at > 0 && --g_fail_at == 0) return 2;
  if (device && g_fail_above > 0 && (long long)bytes > g_fail_above) return 2;
  for (Block &b : g_blocks)
    if (!b.p) {
      b = {(char *)std::calloc(bytes ? bytes : 1, 1), bytes, device};
      if (!b.p) return 2;
      (device ? g_live : g_host_live) += (long long)bytes;
      *p = b.p;
      return 0;
    }
  return 2;
}

int release(void *p)
{
  if (!p) return 0;
  std::lock_guard<std::recursive_mutex> lock(g_mu);
  for (Block &b : g_blocks)
    if (b.p == p) {
      (b.device ? g_live : g_host_live) -= (long long)b.bytes;
      std::free(b.p);
      b = {};
      return 0;
    }
  return 1;
}

void *take(size_t n)
{
  if (g_count_news) {
    ++g_news;
    if (g_fail_new > 0 && --g_fail_new == 0) return nullptr;
  }
  return std::malloc(n ? n : 1);
}

}  // namespace

void *operator new(size_t n)
{
  void *p = take(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void *operator new[](size_t n) { return ::operator new(n); }
void *operator new(size_t n, const std::nothrow_t &) noexcept { return take(n); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete[](void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
void operator delete[](void *p, size_t) noexcept { std::free(p); }

extern "C" {

// ---- what a test asks of it -------------------------------------------------
void stand_in_reset()
{
  std::lock_guard<std::recursive_mutex> lock(g_mu);
  g_nlog = 0;
  g_fail_at = g_fail_above = g_fail_new = 0;
  g_device_allocs = g_host_allocs = g_graph_launches = 0;
  g_news = g_syncs = 0;
}
void stand_in_fail_at(long long n) { g_fail_at = n; }             // the n-th device allocation from here
void stand_in_fail_above(long long bytes) { g_fail_above = bytes; }  // device allocations beyond this size
void stand_in_news(int count, long long fail_at)                  // this thread's operator new
{
  g_news = 0;
  g_count_news = count != 0;
  g_fail_new = fail_at;
}
long long stand_in_value(int what)
{
  const long long v[] = {g_device_allocs, g_host_allocs, g_live, g_news.load(), g_syncs.load(),
                         g_graph_launches, g_copies.load(), g_host_live};
  return v[what];
}
void stand_in_cost(const char *kernel, double us)  // of a launch whose name holds `kernel` (others 1)
{
  std::free((void *)g_slow);
  g_slow = strdup(kernel);
  g_slow_cost = us;
}
int stand_in_launches(const char *kernel)
{
  int n = 0;
  for (int q = 0; q < g_nlog; ++q) n += std::strstr(g_names[g_log[q].name].name, kernel) != nullptr;
  return n;
}

int stand_in_grid(const char *kernel)  // work-groups along x of its last launch
{
  for (int q = g_nlog; q-- > 0;)
    if (std::strstr(g_names[g_log[q].name].name, kernel)) return (int)g_log[q].grid;
  return 0;
}

// ---- the runtime ------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) { return (void **)&g_clock; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
  if (g_nnames < kNames) g_names[g_nnames++] = {host, name};
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
struct dim3s {
  unsigned x, y, z;
};
int __hipPushCallConfiguration(dim3s g, dim3s b, size_t shm, void *stream)
{
  g_config = {{g.x, g.y, g.z}, {b.x, b.y, b.z}, shm, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3s *g, dim3s *b, size_t *shm, void **stream)
{
  *g = {g_config.g[0], g_config.g[1], g_config.g[2]};
  *b = {g_config.b[0], g_config.b[1], g_config.b[2]};
  *shm = g_config.shm;
  *stream = g_config.stream;
  return 0;
}
int hipLaunchKernel(const void *f, dim3s grid, dim3s, void **, size_t, void *)
{
  std::lock_guard<std::recursive_mutex> lock(g_mu);
  for (int q = 0; q < g_nnames; ++q)
    if (g_names[q].host == f) {
      if (!g_capturing) {
        if (g_nlog < kLog) g_log[g_nlog++] = {q, grid.x};
        g_clock += g_slow && std::strstr(g_names[q].name, g_slow) ? g_slow_cost : 1.0;
      }
      return 0;
    }
  return 1;
}
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 8, 0; }
int hipGetSymbolAddress(void **p, const void *)
{
  static char *block = (char *)std::calloc((size_t)32 << 20, 1);
  return *p = block, 0;
}
int hipMalloc(void **p, size_t bytes) { return allocate(p, bytes, true); }
int hipFree(void *p) { return release(p); }
int hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(p, bytes, false); }
int hipHostFree(void *p) { return release(p); }
int hipPointerGetAttributes(int *attr, const void *p)  // its first word is the type: 0 unregistered, 1 host, 2 device
{
  std::lock_guard<std::recursive_mutex> lock(g_mu);
  attr[0] = 0;
  for (const Block &b : g_blocks)
    if (b.p && (const char *)p >= b.p && (const char *)p < b.p + b.bytes) attr[0] = b.device ? 2 : 1;
  return 0;
}
int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int, void *)
{
  ++g_copies;
  if (bytes <= kLargest) std::memcpy(dst, src, bytes);
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t bytes, void *)
{
  if (bytes <= kLargest) std::memset(p, v, bytes);
  return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned) { return *s = std::malloc(8), 0; }
int hipStreamDestroy(void *s) { return std::free(s), 0; }
int hipStreamSynchronize(void *) { return ++g_syncs, 0; }
int hipStreamBeginCapture(void *, int) { return g_capturing = true, 0; }
int hipStreamEndCapture(void *, void **g) { return g_capturing = false, *g = std::malloc(8), 0; }
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) { return *e = std::malloc(8), 0; }
int hipGraphLaunch(void *, void *) { return ++g_graph_launches, 0; }
int hipGraphDestroy(void *g) { return std::free(g), 0; }
int hipGraphExecDestroy(void *e) { return std::free(e), 0; }
int hipEventCreate(void **e) { return *e = std::calloc(1, sizeof(Event)), 0; }
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *e) { return std::free(e), 0; }
int hipEventRecord(void *e, void *) { return ((Event *)e)->at = g_clock, 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b)
{
  *ms = (float)((((Event *)b)->at - ((Event *)a)->at) * 1e-3);
  return 0;
}

}  // extern "C"

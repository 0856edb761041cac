// A stand-in for the HIP runtime that runs nothing and keeps account of order:
// which operation is sure to have ended before which, by the stream it is on,
// the events it waits for and the host's synchronisations (the null stream and
// the library's non-blocking streams do not wait for each other).  It counts
//  * fills and copies into memory that another stream's fill or copy, not sure
//    to have ended, also writes;
//  * launches whose workgroups wait for each other (the synthetic solve's inner
//    loops) that another such launch may run beside;
//  * fills captured into a graph;
// and notes the shortest copy to host memory that is not pinned, and what the
// library itself allocates on the host.
// Loaded with RTLD_GLOBAL before the library, so that it takes the runtime's place.
#include <dlfcn.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {
struct Dim3 { uint32_t x, y, z; };
using Clock = std::map<const void *, long>;  // by stream: the number of its operations that have ended
void join(Clock &a, const Clock &b) {
  for (const auto &e : b) a[e.first] = std::max(a[e.first], e.second);
}
struct Stream { long ops = 0; Clock known; bool capturing = false, gang = false; };
struct Done { const void *stream; long op; };
struct Write { uintptr_t from, to; Done by; };
struct Launch { std::string name; Dim3 grid; };

std::recursive_mutex mu;
std::map<const void *, Stream> streams;  // (the null stream too)
Clock host;                              // what the host knows to have ended
std::map<const void *, Clock> events;
std::vector<Write> writes;
std::vector<Done> gangs;
std::vector<Launch> launches;
std::map<const void *, std::string> kernels;
std::map<void *, size_t> sizes;
std::map<char *, size_t> pinned;
size_t shortest_pageable = SIZE_MAX;
int races = 0, beside = 0, captured_fills = 0, queued = 0, cus = 256;
struct Config { Dim3 g, b; size_t sh; void *s; };
thread_local Config config;
thread_local int last_error = 0;  // (of a call that failed, until it is asked for)
bool no_pinned = false;

Done issue(const void *s) {
  Stream &q = streams[s];
  join(q.known, host);
  return {s, ++q.ops};
}
bool ended_before(const Done &a, const Done &b) {
  return a.stream == b.stream || streams[b.stream].known[a.stream] >= a.op;
}
void wait_for(const void *s) {
  join(host, streams[s].known);
  host[s] = streams[s].ops;
}
void write(void *dst, size_t n, const void *s) {
  if (streams[s].capturing) captured_fills++;
  const Done me = issue(s);
  const uintptr_t a = (uintptr_t)dst, z = a + n;
  for (const Write &w : writes)
    if (w.from < z && a < w.to && !ended_before(w.by, me)) races++;
  writes.push_back({a, z, me});
}
void gang(const void *s) {
  const Done me = issue(s);
  int ahead = 1;
  for (const Done &g : gangs) {
    if (!ended_before(g, me)) beside++;
    ahead += host[g.stream] < g.op;
  }
  queued = std::max(queued, ahead);
  gangs.push_back(me);
}
void launch(const void *f, Dim3 g, const void *s) {
  const std::string &n = kernels[f];
  launches.push_back({n, g});
  const bool is_gang = n.find("k_ns_loop") != std::string::npos || n.find("k_ns_batch") != std::string::npos;
  if (streams[s].capturing) streams[s].gang |= is_gang;
  else if (is_gang) gang(s);
  else (void)issue(s);
}
}  // namespace
// allocations of host memory by the library's own code
static std::atomic<long> own_allocations{0};
__attribute__((noinline)) void *operator new(size_t n) {
  Dl_info info;
  if (dladdr(__builtin_return_address(0), &info) && info.dli_fname && strstr(info.dli_fname, "libgsis")) own_allocations++;
  if (void *p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

#define LOCK std::lock_guard<std::recursive_mutex> lock(mu)

extern "C" {
// ---- the account
long model_own_allocations() { return own_allocations; }
int model_races() { return races; }
int model_beside() { return beside; }
int model_captured_fills() { return captured_fills; }
int model_queued() { return queued; }  // of those launches, the most that the host did not know to have ended
void model_set_cus(int n) { cus = n; }
void model_no_pinned_memory() { no_pinned = true; }
size_t model_shortest_pageable_read() { return shortest_pageable; }
// launches of the kernels whose name contains part; the last one's workgroups
int model_launches(const char *part, int *workgroups) {
  int n = 0;
  for (const Launch &l : launches)
    if (l.name.find(part) != std::string::npos) { n++; *workgroups = (int)l.grid.x; }
  return n;
}

// ---- the runtime's calls
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { kernels[f] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void *s) { config = {g, b, sh, s}; return 0; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *sh, void **s) { *g = config.g; *b = config.b; *sh = config.sh; *s = config.s; return 0; }
int hipLaunchKernel(const void *f, Dim3 g, Dim3, void **, size_t, void *s) { LOCK; launch(f, g, s); return 0; }
int hipLaunchCooperativeKernel(const void *f, Dim3 g, Dim3, void **, unsigned, void *s) { LOCK; launch(f, g, s); return (int)g.x <= cus ? 0 : 720; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = cus; return 0; }  // (asked for the CUs, and for an LDS size that these tests do not reach)
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
const char *hipGetErrorString(int) { return "error of the model"; }
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
int hipGetSymbolAddress(void **, const void *) { return 1; }
int hipMalloc(void **p, size_t n) {  // an address range that nothing reads or writes
  LOCK;
  *p = mmap(nullptr, n, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) return 2;
  sizes[*p] = n;
  return 0;
}
int hipFree(void *p) {
  LOCK;
  for (auto &s : streams) wait_for(s.first);
  const uintptr_t a = (uintptr_t)p, z = a + sizes[p];
  writes.erase(std::remove_if(writes.begin(), writes.end(), [&](const Write &w) { return w.from < z && a < w.to; }), writes.end());
  munmap(p, sizes[p]);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) { LOCK; if (no_pinned) return last_error = 2; *p = malloc(n); pinned[(char *)*p] = n; return 0; }
int hipHostFree(void *p) { LOCK; pinned.erase((char *)p); free(p); return 0; }
int hipMemset(void *p, int, size_t n) { LOCK; write(p, n, nullptr); return 0; }
int hipMemsetD32(void *p, int, size_t n) { LOCK; write(p, 4 * n, nullptr); return 0; }
int hipMemsetAsync(void *p, int, size_t n, void *s) { LOCK; write(p, n, s); return 0; }
static int copy(void *dst, size_t n, int kind, const void *s) {
  LOCK;
  if (kind == 2) {  // to the host: zeros
    auto p = pinned.upper_bound((char *)dst);
    if (p == pinned.begin() || (char *)dst + n > (--p)->first + p->second) shortest_pageable = std::min(shortest_pageable, n);
    memset(dst, 0, n);
    (void)issue(s);
  }
  else write(dst, n, s);
  return 0;
}
int hipMemcpy(void *dst, const void *, size_t n, int kind) { LOCK; copy(dst, n, kind, nullptr); wait_for(nullptr); return 0; }
int hipMemcpyAsync(void *dst, const void *, size_t n, int kind, void *s) { return copy(dst, n, kind, s); }
int hipStreamCreateWithFlags(void **s, unsigned) { LOCK; *s = malloc(1); return 0; }
int hipStreamDestroy(void *) { return 0; }  // (its address is not used again)
int hipStreamSynchronize(void *s) { LOCK; wait_for(s); return 0; }
int hipDeviceSynchronize() { LOCK; for (auto &s : streams) wait_for(s.first); return 0; }
int hipEventCreate(void **e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = malloc(1); return 0; }
int hipEventDestroy(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 1.0f; return 0; }
int hipEventRecord(void *e, void *s) {
  LOCK;
  Clock c = streams[s].known;
  c[s] = streams[s].ops;
  events[e] = c;
  return 0;
}
int hipEventSynchronize(void *e) { LOCK; join(host, events[e]); return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned) { LOCK; join(streams[s].known, events[e]); return 0; }
int hipStreamBeginCapture(void *s, int) { LOCK; streams[s].capturing = true; streams[s].gang = false; return 0; }
int hipStreamEndCapture(void *s, void **g) { LOCK; streams[s].capturing = false; *g = new bool(streams[s].gang); return 0; }
int hipGraphInstantiate(void **x, void *g, void *, char *, size_t) { *x = new bool(*(bool *)g); return 0; }
int hipGraphLaunch(void *x, void *s) { LOCK; if (*(bool *)x) gang(s); else (void)issue(s); return 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
}

// A HIP runtime without a device for tests of the host code: memory is the host's, kernels do not run, work on a stream is
// done when something waits for it, and any call can be made to fail.  Loaded ahead of the library under test, its
// functions take the place of libamdhip64's.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Event {
  hipStream_t stream = nullptr;
  long seq = 0;
};
std::map<hipStream_t, long> g_queued, g_done;
std::map<const void*, std::string> g_names;
std::map<std::string, int> g_calls;
std::string g_fail_name, g_log;
int g_fail_nth = 0;
hipError_t g_last = hipSuccess;
dim3 g_grid, g_block;
hipStream_t g_launch_stream;
size_t g_lds;
int g_selected = 0;

bool fails(const char* name) {
  const int n = ++g_calls[name];
  if (g_fail_name != name || g_fail_nth != n) return false;
  g_last = hipErrorUnknown;
  return true;
}
void queue(hipStream_t s) { ++g_queued[s]; }
void finish_all() { g_done = g_queued; }
}  // namespace

extern "C" {
// ---- for the test ----
// From here on the nth call of `name` fails (0: none); the counts start anew.
void fake_arm(const char* name, int nth) {
  g_fail_name = name;
  g_fail_nth = nth;
  g_last = hipSuccess;
  g_calls.clear();
  g_log.clear();
  finish_all();
}
int fake_calls(const char* name) { return g_calls[name]; }
// Operations that nothing has waited for, on every stream but `except`.
long fake_pending(void* except) {
  long n = 0;
  for (auto& q : g_queued)
    if (q.first != (hipStream_t)except) n += q.second - g_done[q.first];
  return n;
}
// One line a launch or asynchronous copy.
const char* fake_log() { return g_log.c_str(); }
// The number of columns that the hybrid entry's selection kernels find.
void fake_select(int n) { g_selected = n; }

// ---- the runtime ----
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_grid = grid, g_block = block, g_lds = lds, g_launch_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_grid, *block = g_block, *lds = g_lds, *s = g_launch_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t s) {
  if (fails("hipLaunchKernel")) return g_last;
  queue(s);
  const std::string& name = g_names[f];
  char line[64];
  std::snprintf(line, sizeof(line), " %u %u %u %u\n", grid.x, grid.y, grid.z, block.x);
  g_log += "launch " + name + line;
  if (name.find("scan_counts") != std::string::npos) **(int**)args[2] = g_selected;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  if (fails("hipGetDevice")) return g_last;
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return fails("hipSetDevice") ? g_last : hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  if (fails("hipGetDeviceProperties")) return g_last;
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "injected"; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* fixed = std::calloc(1, size_t(32) << 20);
  *p = fixed;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  if (fails("hipMalloc")) return g_last;
  *p = std::aligned_alloc(256, (n + 255) & ~size_t(255));
  if (*p) std::memset(*p, 0, n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (fails("hipHostMalloc")) return g_last;
  *p = std::aligned_alloc(4096, (n + 4095) & ~size_t(4095));
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {  // waits for the device
  finish_all();
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  finish_all();
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  if (fails("hipMemset")) return g_last;
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  if (fails("hipMemcpy")) return g_last;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
  if (fails("hipMemcpyAsync")) return g_last;
  std::memcpy(d, s, n);
  queue(st);
  char line[64];
  std::snprintf(line, sizeof(line), "copy %s %zu\n", kind == hipMemcpyHostToDevice ? "in" : "out", n);
  g_log += line;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  if (fails("hipDeviceSynchronize")) return g_last;
  finish_all();
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  if (fails("hipStreamCreateWithFlags")) return g_last;
  *s = (hipStream_t) new char;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  g_queued.erase(s), g_done.erase(s);
  delete (char*)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (fails("hipStreamSynchronize")) return g_last;
  g_done[s] = g_queued[s];
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return fails("hipStreamWaitEvent") ? g_last : hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (fails("hipEventCreateWithFlags")) return g_last;
  *e = (hipEvent_t) new Event;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (fails("hipEventRecord")) return g_last;
  *(Event*)e = Event{s, g_queued[s]};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (fails("hipEventSynchronize")) return g_last;
  const Event& v = *(Event*)e;
  if (g_done[v.stream] < v.seq) g_done[v.stream] = v.seq;
  return hipSuccess;
}
}

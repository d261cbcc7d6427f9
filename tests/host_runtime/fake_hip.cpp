// A stand-in for the HIP runtime, so that the library's host code runs where there is no device: two devices whose memory is the
// host's, streams that hold their work back until somebody waits for it, and the runtime's own rules about
// which device an object belongs to.  Of the kernels only the byte copy does anything.  Built and loaded by
// tests/test_host_runtime.py in place of libamdhip64.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
std::recursive_mutex mu;
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
std::map<const void*, std::string> kernels;
std::map<std::string, long> launched;
std::string launches;  // the names of all launches, in order, one a line
std::map<uintptr_t, std::pair<size_t, int>> pinned;  // pinned host memory: bytes, device
size_t refused_bytes = 0;  // allocations of exactly this size fail

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
bool is_pinned(const void* p) {
  auto it = pinned.upper_bound((uintptr_t)p);
  return it != pinned.begin() && (uintptr_t)p < (--it)->first + it->second.first;
}
}  // namespace

struct ihipStream_t {
  int device;
  std::deque<std::function<void()>> work;
  uint64_t queued = 0, done = 0;
  void add(std::function<void()> f) { work.push_back(std::move(f)), queued++; }
  void run_to(uint64_t n) {
    while (done < n) work.front()(), work.pop_front(), done++;
  }
};
struct ihipEvent_t {
  int device;
  ihipStream_t* stream = nullptr;
  uint64_t at = 0;
};

// held by every call that changes something; `inside`: the runtime's own allocations are not the ones to fail
thread_local int inside = 0;
long failing_new = -1;  // operator new calls left until the one that fails
struct Locked {
  Locked() { mu.lock(), inside++; }
  ~Locked() { inside--, mu.unlock(); }
};
#define LOCK Locked lock

void* operator new(size_t n) {
  if (!inside) {
    LOCK;
    if (failing_new >= 0 && failing_new-- == 0) throw std::bad_alloc();
  }
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
void fake_refuse_allocations_of(size_t bytes) { refused_bytes = bytes; }
void fake_fail_allocation(long n) { failing_new = n; }
const char* fake_launch_log() {  // since the last time it was asked for
  LOCK;
  static std::string given;
  return given.swap(launches), launches.clear(), given.c_str();
}
long fake_launches(const char* part_of_name) {
  LOCK;
  long n = 0;
  for (auto& k : launched)
    if (k.first.find(part_of_name) != std::string::npos) n += k.second;
  return n;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipSetDevice(int d) { return current = d, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = current, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  return last = hipSuccess, e;
}
hipError_t hipMalloc(void** p, size_t n) {
  if (n == refused_bytes) return ret(hipErrorOutOfMemory);
  return *p = std::aligned_alloc(256, (n + 255) & ~(size_t)255), *p ? hipSuccess : ret(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  LOCK;
  *p = std::aligned_alloc(4096, (n + 4095) & ~(size_t)4095);
  pinned[(uintptr_t)*p] = {n, current};
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  LOCK;
  pinned.erase((uintptr_t)p), std::free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  LOCK;
  std::memset(a, 0, sizeof *a);
  a->type = is_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), hipSuccess; }

hipError_t hipStreamCreate(hipStream_t* s) {
  LOCK;
  return *s = new ihipStream_t{current, {}}, hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  LOCK;
  s->run_to(s->queued);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
  LOCK;
  return s->done == s->queued ? hipSuccess : ret(hipErrorNotReady);
}
hipError_t hipStreamDestroy(hipStream_t s) {
  hipStreamSynchronize(s);
  delete s;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  LOCK;
  return *e = new ihipEvent_t{current}, hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  LOCK;
  if (e->device != s->device) return ret(hipErrorInvalidHandle);  // as the runtime does
  e->stream = s, e->at = s->queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  LOCK;
  if (e->stream) e->stream->run_to(e->at);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }

hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  LOCK;
  s->add([=] { std::memset(p, v, n); });
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* src, size_t n, hipMemcpyKind kind, hipStream_t s) {
  LOCK;
  s->add([=] { std::memcpy(d, src, n); });
  const void* const host = kind == hipMemcpyHostToDevice ? src : kind == hipMemcpyDeviceToHost ? d : nullptr;
  if (host && !is_pinned(host)) s->run_to(s->queued);  // pageable memory is staged before the call returns
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t s) {
  LOCK;
  const std::string& name = kernels[f];
  launched[name]++;
  launches += name + " " + std::to_string(grid.x) + " " + std::to_string(grid.y) + " " + std::to_string(grid.z) + " " + std::to_string(block.x) + "\n";
  if (name.find("copy_bytes_kernel") != std::string::npos) {
    void *dst = *(void**)args[0], *src = *(void**)args[1];
    const size_t n = (size_t)*(uint32_t*)args[2] * 16 + *(uint32_t*)args[3];
    s->add([=] { std::memcpy(dst, src, n); });
  }
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
static thread_local dim3 pushed_grid, pushed_block;
static thread_local size_t pushed_lds;
static thread_local hipStream_t pushed_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
  return pushed_grid = g, pushed_block = b, pushed_lds = l, pushed_stream = s, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
  return *g = pushed_grid, *b = pushed_block, *l = pushed_lds, *s = pushed_stream, hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels[f] = name; }
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return ret(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return ret(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return ret(hipErrorNotSupported); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return ret(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// A HIP runtime in host memory for the tests of the engine's host code: device
// memory up to a limit, streams and events that know their device, kernels
// that do nothing.  Loaded ahead of libxfdtd_hip.so (RTLD_GLOBAL), whose calls
// then come here.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {

std::mutex m;
std::map<char*, size_t> blocks;
size_t used = 0, limit = size_t(1) << 40, launches = 0;
int devices = 1;
thread_local int current = 0;

// a stream, an event, a graph: an object of a device
struct Object {
  int device;
};
void* object() { return new Object{current}; }
int forget(void* p) {
  delete static_cast<Object*>(p);
  return 0;
}
int on(void* p) { return p ? static_cast<Object*>(p)->device : current; }

[[noreturn]] void bad(const char* what) {
  std::fprintf(stderr, "fake HIP: %s\n", what);
  std::abort();
}

// a range that begins in device memory has to end in the same block; memory
// that was freed is no host memory either
void check(const void* at, size_t n) {
  std::lock_guard<std::mutex> lock(m);
  char* p = static_cast<char*>(const_cast<void*>(at));
  auto it = blocks.upper_bound(p);
  if (it == blocks.begin()) return;
  --it;
  if (p < it->first + it->second && p + n > it->first + it->second) bad("copy past the end of an allocation");
}

}  // namespace

extern "C" {

void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_used() { return used; }
size_t fake_launches() { return launches; }
void fake_devices(int n) { devices = n; }

int hipGetDeviceCount(int* n) {
  *n = devices;
  return 0;
}
int hipSetDevice(int d) {
  current = d;
  return 0;
}
int hipGetLastError() { return 0; }
int hipDeviceSynchronize() { return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : e == 400 ? "invalid handle" : "fake error"; }

int hipMemGetInfo(size_t* free_bytes, size_t* all) {
  std::lock_guard<std::mutex> lock(m);
  *free_bytes = limit > used ? limit - used : 0;
  *all = limit;
  return 0;
}
int hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lock(m);
  if (used + n > limit) return 2;
  *p = std::malloc(n ? n : 1);
  blocks[static_cast<char*>(*p)] = n;
  used += n;
  return 0;
}
int hipFree(void* p) {
  if (!p) return 0;
  std::lock_guard<std::mutex> lock(m);
  const auto it = blocks.find(static_cast<char*>(p));
  if (it == blocks.end()) bad("free of what is not allocated");
  std::memset(p, 0xa5, it->second);
  used -= it->second;
  blocks.erase(it);
  std::free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return 0;
}
int hipHostFree(void* p) {
  std::free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  check(d, n);
  check(s, n);
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) { return hipMemcpy(d, s, n, kind); }
int hipMemset(void* d, int v, size_t n) {
  check(d, n);
  std::memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }

int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = object();
  return 0;
}
int hipStreamDestroy(void* s) { return forget(s); }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
  *g = object();
  return 0;
}
int hipGraphDestroy(void* g) { return forget(g); }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
  *x = object();
  return 0;
}
int hipGraphExecDestroy(void* x) { return forget(x); }
int hipGraphLaunch(void* x, void*) { return x ? 0 : 400; }

int hipEventCreate(void** e) {
  *e = object();
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { return forget(e); }
// an event is recorded on a stream of its own device
int hipEventRecord(void* e, void* s) { return on(e) == on(s) ? 0 : 400; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 1.0f;
  return 0;
}

int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipGetDevicePropertiesR0600(void* p, int) {
  std::memset(p, 0, 1472);  // sizeof(hipDeviceProp_tR0600)
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return 0;
}
int hipGetSymbolAddress(void**, const void*) { return 1; }

int __hipPushCallConfiguration(unsigned long, unsigned, unsigned long, unsigned, size_t, void*) { return 0; }
int __hipPopCallConfiguration(void*, void*, size_t*, void**) { return 0; }
int hipLaunchKernel(const void*, unsigned long, unsigned, unsigned long, unsigned, void**, size_t, void*) {
  std::lock_guard<std::mutex> lock(m);
  ++launches;
  return 0;
}

}  // extern "C"

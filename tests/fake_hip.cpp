// A HIP runtime on host memory, for tests of the library's host code without a
// GPU: loaded before libhes.so, its functions stand in for the runtime's.
// Device memory is host memory, a launch runs nothing except the kernels that
// move a state in and out (named below), and allocations can be made to fail,
// the library's own of host memory among them.
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
constexpr int OK = 0, OUT_OF_MEMORY = 2;
std::mutex mutex;
std::map<const void*, std::string> kernels;
std::map<std::string, long long> launches;
std::map<void*, size_t> device;
size_t device_used = 0, device_cap = ~(size_t)0, device_fail_min = ~(size_t)0;
size_t host_fail_min = ~(size_t)0;
long long host_allowed = 0;  // host allocations of at least host_fail_min that still succeed
std::atomic<bool> new_fails{false};
thread_local int inside = 0;  // this file's own allocations always succeed
struct Lock {
  std::lock_guard<std::mutex> lock{mutex};
  Lock() { ++inside; }
  ~Lock() { --inside; }
};
thread_local int last_error = OK;
int result(int e) {
  if (e != OK) last_error = e;
  return e;
}
struct Dim3 {
  uint32_t x, y, z;
};
struct Config {
  Dim3 grid, block;
  size_t shared;
  void* stream;
};
thread_local Config config;
}  // namespace

void* operator new(size_t n) {
  void* p = new_fails && !inside ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
// ---- what a test sets and reads
void fake_new_fails(int on) { new_fails = on != 0; }  // the library's own allocations of host memory
void fake_device_cap(size_t bytes) { device_cap = bytes; }
void fake_device_fail_from(size_t bytes) { device_fail_min = bytes; }  // allocations this large fail
void fake_host_fail_from(size_t bytes, long long allowed) {
  host_fail_min = bytes;
  host_allowed = allowed;
}
long long fake_launches(const char* name) {  // of kernels whose name contains this
  Lock lock;
  long long n = 0;
  for (auto& k : launches)
    if (k.first.find(name) != std::string::npos) n += k.second;
  return n;
}
size_t fake_device_used() { return device_used; }

// ---- the runtime
int hipMalloc(void** p, size_t n) {
  Lock lock;
  if (n >= device_fail_min || device_used + n > device_cap) return result(OUT_OF_MEMORY);
  *p = std::calloc(1, n ? n : 1);
  device[*p] = n;
  device_used += n;
  return OK;
}
int hipFree(void* p) {
  Lock lock;
  if (p) {
    device_used -= device[p];
    device.erase(p);
    std::free(p);
  }
  return OK;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  Lock lock;
  if (n >= host_fail_min && host_allowed-- <= 0) return result(OUT_OF_MEMORY);
  *p = std::calloc(1, n);
  return OK;
}
int hipHostFree(void* p) { std::free(p); return OK; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return OK; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); return OK; }
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return OK; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { std::memset(d, v, n); return OK; }
int hipGetDevice(int* d) { *d = 0; return OK; }
int hipSetDevice(int) { return OK; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return OK; }
int hipGetLastError() {
  const int e = last_error;
  last_error = OK;
  return e;
}
const char* hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "no error"; }
int hipFuncGetAttributes(void* attributes, const void*) {  // 5 ints, 3 sizes, padding: all 0
  std::memset(attributes, 0, 56);
  return OK;
}
int hipFuncSetAttribute(const void*, int, int) { return OK; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = std::malloc(1); return OK; }
int hipStreamDestroy(void* s) { std::free(s); return OK; }
int hipStreamSynchronize(void*) { return OK; }
int hipStreamBeginCapture(void*, int) { return OK; }
int hipStreamEndCapture(void*, void** g) { *g = std::malloc(1); return OK; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = std::malloc(1); return OK; }
int hipGraphLaunch(void*, void*) { return OK; }
int hipGraphDestroy(void* g) { std::free(g); return OK; }
int hipGraphExecDestroy(void* x) { std::free(x); return OK; }
int hipStreamWaitEvent(void*, void*, unsigned) { return OK; }
int hipEventCreate(void** e) { *e = std::malloc(1); return OK; }
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { std::free(e); return OK; }
int hipEventRecord(void*, void*) { return OK; }
int hipEventSynchronize(void*) { return OK; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.f; return OK; }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*,
                           void*, int*) {
  Lock lock;
  kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  config = {grid, block, shared, stream};
  return OK;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return OK;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void** a, size_t, void*) {
  std::string name;
  {
    Lock lock;
    name = kernels[f];
    ++launches[name];
  }
  auto ll = [&](int k) { return *(long long*)a[k]; };
  if (name.find("k_aos_to_soa") != std::string::npos) {  // in, out, nc, n, pitch
    const double* in = *(const double**)a[0];
    double* out = *(double**)a[1];
    const int nc = *(int*)a[2];
    for (long long i = 0; i < ll(3); ++i)
      for (int r = 0; r < nc; ++r) out[r * ll(4) + i] = in[i * nc + r];
  } else if (name.find("k_gather") != std::string::npos) {  // Q, out, nc, first, cells, pitch
    const double* q = *(const double**)a[0];
    double* out = *(double**)a[1];
    const int nc = *(int*)a[2];
    for (long long i = 0; i < ll(4); ++i)
      for (int r = 0; r < nc; ++r) out[i * nc + r] = q[r * ll(5) + ll(3) + i];
  }
  return OK;
}
}

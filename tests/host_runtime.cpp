// The HIP runtime calls of libolive_hip.so on host memory, for tests of the
// library's host code without a GPU.  Preloaded, it answers allocations from
// the heap, copies with memcpy and hands every kernel launch to a callback (by
// kernel name) instead of running it; a chosen allocation can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Config {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
};
std::map<const void *, std::string> &kernels() {
  static std::map<const void *, std::string> m;
  return m;
}
std::map<void *, size_t> &blocks() {
  static std::map<void *, size_t> m;
  return m;
}
std::vector<Config> g_config;
void (*g_hook)(const char *name, unsigned grid, void **args) = nullptr;
long g_allocs = 0, g_fail_at = 0;  // allocations so far; the one to fail (0: none)
hipError_t g_last = hipSuccess;    // kept until hipGetLastError reports it
size_t g_live = 0;

hipError_t allocate(void **p, size_t bytes) {
  *p = nullptr;
  if (++g_allocs == g_fail_at) return g_last = hipErrorOutOfMemory;
  *p = std::calloc(1, bytes ? bytes : 1);
  if (!*p) return hipErrorOutOfMemory;
  blocks()[*p] = bytes;
  g_live += bytes;
  return hipSuccess;
}
hipError_t release(void *p) {
  if (!p) return hipSuccess;
  auto it = blocks().find(p);
  if (it == blocks().end()) std::abort();  // not an allocation of this runtime, or freed twice
  g_live -= it->second;
  blocks().erase(it);
  std::free(p);
  return hipSuccess;
}
}  // namespace

extern "C" {
void rt_hook(void (*f)(const char *, unsigned, void **)) { g_hook = f; }
void rt_fail_at(long n) { g_allocs = 0, g_fail_at = n; }  // the n-th allocation from here on
long rt_allocs() { return g_allocs; }
size_t rt_live() { return g_live; }

void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
  kernels()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
  g_config.push_back(Config{grid, block, shmem, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *stream) {
  const Config c = g_config.back();
  g_config.pop_back();
  *grid = c.grid, *block = c.block, *shmem = c.shmem, *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t) {
  if (g_hook) g_hook(kernels()[f].c_str(), grid.x, args);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) { return allocate(p, bytes); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(p, bytes); }
hipError_t hipFree(void *p) { return release(p); }
hipError_t hipHostFree(void *p) { return release(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = reinterpret_cast<hipEvent_t>(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  return g_last = hipSuccess, e;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char scratch[size_t(32) << 20];
  return *p = scratch, hipSuccess;
}
}

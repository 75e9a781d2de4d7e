// A HIP runtime without a device, for tests of the library's host code: device
// memory is host memory, copies are copies, a launch runs nothing and is
// written down.  Loaded before the library, its functions take the place of
// the runtime's.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Launch {
  std::string name;
  void *ptr[2];  // pointer arguments 1 and 2 of the batch kernels, else null
};
std::map<const void *, std::string> g_kernels;
std::vector<Launch> g_launches;
std::map<void *, size_t> g_live;
long g_mallocs = 0, g_fail_at = 0, g_pointer_queries = 0, g_busy = 0;
float g_elapsed = 1e6f;
hipError_t g_last = hipSuccess;
char g_symbol[1 << 20];

hipError_t take(void **p, size_t bytes) {
  *p = std::calloc(bytes ? bytes : 1, 1);
  g_live[*p] = bytes;
  return hipSuccess;
}

}  // namespace

extern "C" {

// --- what the tests ask for ---
long host_mallocs() { return g_mallocs; }
void host_fail_malloc(long nth) {  // the nth allocation from now on fails; 0: none
  g_mallocs = 0;
  g_fail_at = nth;
}
long host_pointer_queries() { return g_pointer_queries; }
void host_busy(long n) { g_busy = n; }  // the stream is at work for the next n queries
long host_live() { return (long)g_live.size(); }
void host_forget() { g_launches.clear(); }
long host_launches() { return (long)g_launches.size(); }
const char *host_launch_name(long k) { return g_launches[k].name.c_str(); }
void *host_launch_ptr(long k, int q) { return g_launches[k].ptr[q]; }

// --- the runtime ---
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static dim3 g_grid, g_block;
static size_t g_shm;
static hipStream_t g_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  g_grid = g;
  g_block = b;
  g_shm = m;
  g_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
  *g = g_grid;
  *b = g_block;
  *m = g_shm;
  *s = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
  Launch l{g_kernels[f], {nullptr, nullptr}};
  if (l.name.find("k_batch_") != std::string::npos)
    for (int q = 0; q < 2; q++) l.ptr[q] = *(void **)args[q + 1];
  g_launches.push_back(l);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
  if (++g_mallocs == g_fail_at) {
    *p = nullptr;
    return g_last = hipErrorOutOfMemory;
  }
  return take(p, bytes);
}
hipError_t hipFree(void *p) {
  if (p && !g_live.erase(p)) return hipErrorInvalidValue;
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return take(p, bytes); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = g_symbol;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  g_pointer_queries++;
  std::memset(a, 0, sizeof(*a));
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipEventCreate(hipEvent_t *e) { return take((void **)e, 8); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipFree(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// ever shorter, so that the form a tuner times last is the one it picks
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = g_elapsed *= 0.999f;
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return take((void **)s, 8); }
hipError_t hipStreamDestroy(hipStream_t s) { return hipFree(s); }
hipError_t hipStreamQuery(hipStream_t) {
  if (g_busy <= 0) return hipSuccess;
  g_busy--;
  return g_last = hipErrorNotReady;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  return take((void **)g, 8);
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return take((void **)e, 8);
}
hipError_t hipGraphDestroy(hipGraph_t g) { return hipFree(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return hipFree(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

}  // extern "C"

// A HIP runtime without a device, for CPU tests of the host library: it takes
// the place of libamdhip64 (loaded with RTLD_GLOBAL before the library).
// Memory is addresses and a count of free bytes, copies and kernels do nothing
// but are counted, kernels by name.  As with the runtime, an error stays the
// last error until hipGetLastError returns it.
#include <hip/hip_runtime.h>

#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Fake {
  size_t free = (size_t)256 << 30, total = (size_t)288 << 30;
  size_t malloc_limit = ~(size_t)0;  // hipMalloc of more fails whatever is free
  size_t next = (size_t)1 << 40;
  std::map<size_t, size_t> live;
  hipError_t last = hipSuccess;
  std::string fail_launch;           // kernels whose name contains it are not launched
  long long mallocs = 0, frees = 0, device_syncs = 0, stream_syncs = 0, copies = 0;
  long long copy_bytes = 0;
  long long graph_launches = 0;
  const void *copy_src = nullptr;    // of the last asynchronous copy
  size_t copy_n = 0;
  bool capturing = false;            // every stream but the default one
  std::map<const void *, std::string> names;
  std::vector<const void *> launched;
  dim3 grid, block;
  size_t lds = 0;
  hipStream_t stream = nullptr;
};
Fake &f() {
  static Fake s;
  return s;
}
hipError_t ret(hipError_t e) {
  if (e != hipSuccess) f().last = e;
  return e;
}
template <typename T>
hipError_t handle(T *h) {
  *h = reinterpret_cast<T>(f().next += 256);
  return hipSuccess;
}

}  // namespace

extern "C" {

// ---- the tests' side
void fake_set_free(size_t bytes) { f().free = bytes; }
size_t fake_free() { return f().free; }
void fake_set_malloc_limit(size_t bytes) { f().malloc_limit = bytes; }
void fake_fail_launch(const char *name) { f().fail_launch = name; }
const void *fake_copy_src(size_t *n) {
  *n = f().copy_n;
  return f().copy_src;
}
void fake_set_capturing(int yes) { f().capturing = yes != 0; }
long long fake_count(const char *what) {
  const std::string w = what;
  if (w == "malloc") return f().mallocs;
  if (w == "free") return f().frees;
  if (w == "device_sync") return f().device_syncs;
  if (w == "stream_sync") return f().stream_syncs;
  if (w == "copy") return f().copies;
  if (w == "graph_launch") return f().graph_launches;
  if (w == "copy_bytes") return f().copy_bytes;
  long long n = 0;  // launches of kernels whose name contains it
  for (const void *k : f().launched) n += f().names[k].find(w) != std::string::npos;
  return n;
}

// ---- the library's side
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  f().names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  f().grid = g;
  f().block = b;
  f().lds = lds;
  f().stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = f().grid;
  *b = f().block;
  *lds = f().lds;
  *s = f().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *k, dim3, dim3, void **, size_t, hipStream_t) {
  const std::string &n = f().names[k];
  if (!f().fail_launch.empty() && n.find(f().fail_launch) != std::string::npos)
    return ret(hipErrorLaunchFailure);
  f().launched.push_back(k);
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) {
  if (n > f().free || n > f().malloc_limit) return ret(hipErrorOutOfMemory);
  f().mallocs++;
  f().free -= n;
  *p = reinterpret_cast<void *>(f().next);
  f().live[f().next] = n;
  f().next += (n + 511) / 256 * 256;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = f().live.find(reinterpret_cast<size_t>(p));
  if (it == f().live.end()) return p ? ret(hipErrorInvalidValue) : hipSuccess;
  f().frees++;
  f().free += it->second;
  f().live.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = new char[n];
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  delete[] static_cast<char *>(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *freeb, size_t *totalb) {
  *freeb = f().free;
  *totalb = f().total;
  return hipSuccess;
}
hipError_t hipMemcpy(void *, const void *, size_t n, hipMemcpyKind) {
  f().copies++;
  f().copy_bytes += (long long)n;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
  f().copies++;
  f().copy_src = src;
  f().copy_n = n;
  f().copy_bytes += (long long)n;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  memset(a, 0, sizeof(*a));
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}

hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = reinterpret_cast<void *>((size_t)1 << 39);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = f().last;
  f().last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "fake error"; }

hipError_t hipDeviceSynchronize() {
  f().device_syncs++;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  f().stream_syncs++;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *g, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return handle(g);
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  f().graph_launches++;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  *st = f().capturing && s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}

}  // extern "C"

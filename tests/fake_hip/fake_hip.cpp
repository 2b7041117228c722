// A stand-in for the HIP runtime, for tests of the library's host code without a GPU.  Device and
// pinned memory are host memory, kernels do nothing but the read-back's two, and the test sets what fails and reads what was
// called.  Loaded with RTLD_GLOBAL before libnbgpu.so, its definitions are the ones that the library
// binds to (operator new among them).
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

static std::mutex mu;
static std::map<const void *, std::string> &names() {
  static auto *m = new std::map<const void *, std::string>();
  return *m;
}
static std::string launched;  // names of the kernels launched, one a line
static size_t budget = SIZE_MAX, in_use = 0;
static long host_mallocs = 0, dev_mallocs = 0, dev_copies = 0;
static long publish_pairs = -1;
static std::atomic<long> new_countdown{-1};

static hipError_t last_error = hipSuccess;

struct Head {
  size_t bytes, pad[31];
};

extern "C" {
void fake_budget(size_t bytes) { budget = bytes; }       // device memory left to hipMalloc
size_t fake_in_use() { return in_use; }
long fake_host_mallocs() { return host_mallocs; }
long fake_dev_mallocs() { return dev_mallocs; }
long fake_dev_copies() { return dev_copies; }  // copies from device to device asked of the runtime
// the library's n-th operator new from now (0: the next one) fails, once; -1: none
void fake_fail_new(long n) { new_countdown = n; }
long fake_new_left() { return new_countdown; }
// the number of pairs that the counters read back say (-1: what the device memory holds)
void fake_pairs(long n) { publish_pairs = n; }
void fake_clear() {
  std::lock_guard<std::mutex> l(mu);
  launched.clear();
}
const char *fake_launched() { return launched.c_str(); }

// ---- launches ----
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
void **__hipRegisterFatBinary(const void *) {
  static void *h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  std::lock_guard<std::mutex> l(mu);
  names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st) {
  cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st) {
  *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *st = cfg_stream;
  return hipSuccess;
}
struct PackArgs {  // nb_stage.hip's
  const void *src[16];
  uint32_t bytes[16], at[16];
  char *dst;
};
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t) {
  std::lock_guard<std::mutex> l(mu);
  const std::string &n = names()[f];
  launched += n + "\n";
  // the counters' copy to pinned memory: the first word is the pair count
  if (n.find("k_publish") != std::string::npos) {
    char *dst = *static_cast<char **>(args[1]), *src = *static_cast<char **>(args[0]);
    memcpy(dst, src, (reinterpret_cast<Head *>(src) - 1)->bytes);
    const uint32_t p = publish_pairs;
    if (publish_pairs >= 0) memcpy(dst, &p, sizeof p);
  }
  if (n.find("k_pack") != std::string::npos) {
    const PackArgs &a = *static_cast<PackArgs *>(args[0]);
    for (unsigned c = 0; c < grid.y; c++) memcpy(a.dst + a.at[c], a.src[c], a.bytes[c]);
  }
  return hipSuccess;
}

// ---- memory ----
hipError_t hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> l(mu);
  dev_mallocs++;
  *p = nullptr;
  if (bytes > budget) return last_error = hipErrorOutOfMemory;
  Head *h = static_cast<Head *>(calloc(1, sizeof(Head) + bytes));
  if (!h) return hipErrorOutOfMemory;
  h->bytes = bytes;
  in_use += bytes;
  if (budget != SIZE_MAX) budget -= bytes;
  *p = h + 1;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  std::lock_guard<std::mutex> l(mu);
  Head *h = static_cast<Head *>(p) - 1;
  in_use -= h->bytes;
  if (budget != SIZE_MAX) budget += h->bytes;
  free(h);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  std::lock_guard<std::mutex> l(mu);
  host_mallocs++;
  *p = calloc(1, bytes);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k == hipMemcpyDeviceToDevice) dev_copies++;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = nullptr;
  return hipErrorInvalidSymbol;
}

// ---- devices, streams, events, graphs ----
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  return *n = 2, hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = reinterpret_cast<hipGraph_t>(8);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(8);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// ---- operator new ----
static void *get(size_t n, const void *caller) {
  Dl_info d;
  if (new_countdown >= 0 && dladdr(caller, &d) && strstr(d.dli_fname, "libnbgpu") &&
      new_countdown.fetch_sub(1) == 0)
    return nullptr;
  return malloc(n ? n : 1);
}
#define CALLER __builtin_return_address(0)
void *operator new(size_t n) {
  void *p = get(n, CALLER);
  if (!p) throw std::bad_alloc();
  return p;
}
void *operator new[](size_t n) {
  void *p = get(n, CALLER);
  if (!p) throw std::bad_alloc();
  return p;
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return get(n, CALLER); }
void *operator new[](size_t n, const std::nothrow_t &) noexcept { return get(n, CALLER); }
void operator delete(void *p) noexcept { free(p); }
void operator delete[](void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
void operator delete[](void *p, size_t) noexcept { free(p); }

// nb_stage.hip -- device arrays to caller memory through pinned staging.
//
// The caller's arrays are ordinary memory.  A copy straight into it costs the runtime 15 to 25 us a
// call however small, and large ones run at one thread's page-fault rate: reading back 13 arrays
// took 0.22 ms for 1,000 bodies, 1.8 for 100,003, 5.5 for 262,144 and 12.6 for 1,048,576 (medians),
// a frame of 1,048,576 bodies 1.06 ms.  Here one kernel writes a slice of the arrays to pinned host
// memory over the bus, and up to 8 threads move the slices that have arrived: 0.04, 0.7, 1.6, 2.9
// and 0.39 ms.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

#include "nb_internal.hpp"

namespace nb {

constexpr size_t kStageMax = (size_t)32 << 20;    // bytes of a pinned buffer at most
constexpr size_t kStagePiece = (size_t)1 << 20;   // bytes a thread moves at a time
constexpr size_t kStageSlice = (size_t)4 << 20;   // bytes per launch (and per event)
constexpr size_t kStageSmall = (size_t)1 << 20;   // total up to which one launch and one thread do
constexpr int kStageSlices = 64;                  // slices in flight at most (8 of full size fit)

// Pieces of device arrays to pinned host memory: the kernel's stores go over the bus in whole lines,
// as fast as the copy engine's (about 53 GB/s), and a launch takes up to 16 pieces where a copy call
// takes one.
struct PackArgs {
  const void *src[kFetchMax];
  uint32_t bytes[kFetchMax];
  uint32_t at[kFetchMax];  // offset in dst, a multiple of 16
  char *dst;
};

template <class T>
__device__ __forceinline__ void pack_as(const void *src, char *dst, uint32_t bytes) {
  const T *s = static_cast<const T *>(src);
  T *d = reinterpret_cast<T *>(dst);
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < bytes / sizeof(T); i += gridDim.x * 256)
    d[i] = s[i];
}
__global__ __launch_bounds__(256) void k_pack(PackArgs a) {
  const int c = blockIdx.y;
  const uint32_t bytes = a.bytes[c];
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.src[c]);
  char *dst = a.dst + a.at[c];
  // the widest access that the source's alignment and the size allow
  if (((at | bytes) & 15) == 0) pack_as<uint4>(a.src[c], dst, bytes);
  else if (((at | bytes) & 7) == 0) pack_as<uint2>(a.src[c], dst, bytes);
  else if (((at | bytes) & 3) == 0) pack_as<uint32_t>(a.src[c], dst, bytes);
  else pack_as<uint8_t>(a.src[c], dst, bytes);
}

__global__ void k_publish(const DevCounters *c, DevCounters *host) {
  const uint32_t *s = reinterpret_cast<const uint32_t *>(c);
  uint32_t *d = reinterpret_cast<uint32_t *>(host);
  for (int i = threadIdx.x; i < (int)(sizeof(DevCounters) / 4); i += blockDim.x) d[i] = s[i];
}

// The pinned buffers, with the events recorded beside them.  Allocating one takes the better part
// of a millisecond, so they outlive a context: idle ones wait here, at most kStageIdle of at most
// kStageMax bytes each, and all are freed when the last context, batch or network of the process
// goes.  A buffer belongs to one call at a time, so any number of threads and streams may fetch at
// once.  Its lists have fixed room: the calls are C entries, from which nothing may be thrown.
struct Piece {
  char *dst;
  size_t at, bytes;
  int slice;
};
struct StageBuf {
  int device = 0;
  char *buf = nullptr;
  size_t bytes = 0;
  int nev = 0;
  hipEvent_t ev[kStageSlices];
  Piece window[kStageSlices * kFetchMax];  // a call's pieces, as many as the staging holds
};
constexpr int kStageIdle = 4;
static std::mutex g_mutex;
static StageBuf *g_idle[kStageIdle];
static int g_nidle = 0;
static int g_users = 0;

static void destroy(StageBuf *b) {
  for (int k = 0; k < b->nev; k++) (void)hipEventDestroy(b->ev[k]);
  if (b->buf) (void)hipHostFree(b->buf);
  delete b;
}

void stage_user(int add) {
  StageBuf *gone[kStageIdle];
  int n = 0;
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_users += add;
    if (g_users == 0)
      while (g_nidle > 0) gone[n++] = g_idle[--g_nidle];
  }
  for (int k = 0; k < n; k++) destroy(gone[k]);
}

namespace {
struct Lease {  // a buffer for one call
  StageBuf *b = nullptr;
  void *dev = nullptr;  // its address on the device
  Lease(size_t want) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return;
    {
      std::lock_guard<std::mutex> lock(g_mutex);
      int at = -1;
      for (int k = 0; k < g_nidle; k++)
        if (g_idle[k]->device == device && (at < 0 || g_idle[k]->bytes > g_idle[at]->bytes)) at = k;
      if (at >= 0) {
        b = g_idle[at];
        g_idle[at] = g_idle[--g_nidle];
      }
    }
    if (!b && !(b = new (std::nothrow) StageBuf())) return;
    b->device = device;
    // 1 MiB costs no more than 64 KiB (40 us); an allocation right after a free takes 300, so a
    // buffer grows seldom and the old one goes last
    size_t size = (size_t)1 << 20;
    while (size < want && size < kStageMax) size <<= 1;
    if (size > b->bytes) {
      char *old = b->buf;
      b->buf = nullptr;
      b->bytes = 0;
      if (hipHostMalloc((void **)&b->buf, size, hipHostMallocMapped) == hipSuccess)
        b->bytes = size;
      if (old) (void)hipHostFree(old);
    }
    if (b->bytes == 0 || hipHostGetDevicePointer(&dev, b->buf, 0) != hipSuccess) {
      (void)hipGetLastError();
      destroy(b);
      b = nullptr;
    }
  }
  ~Lease() {
    if (!b) return;
    {
      std::lock_guard<std::mutex> lock(g_mutex);
      if (g_users > 0 && g_nidle < kStageIdle) {
        g_idle[g_nidle++] = b;
        b = nullptr;
      }
    }
    if (b) destroy(b);
  }
  Lease(const Lease &) = delete;
};
}  // namespace

hipError_t stage_counters(const DevCounters *c, hipStream_t st, DevCounters *out) {
  Lease l(sizeof(DevCounters));
  if (!l.b) {
    const hipError_t e = hipMemcpyAsync(out, c, sizeof *out, hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  }
  hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, st, c, (DevCounters *)l.dev);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e == hipSuccess) memcpy(out, l.b->buf, sizeof *out);
  return e;
}

// Slices of host arrays, read by the kernel over the bus.
struct SendArgs {
  void *dst[kFetchMax];
  uint32_t at[kFetchMax];  // offset in src
  int width[kFetchMax];
  const char *src;
  int count;
};
__global__ __launch_bounds__(256) void k_send_reversed(SendArgs a) {
  const int c = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x, j = a.count - 1 - i;
  if (j < 0) return;
  const char *s = a.src + a.at[c];
  if (a.width[c] == 8) static_cast<uint64_t *>(a.dst[c])[j] = ((const uint64_t *)s)[i];
  else if (a.width[c] == 4) static_cast<uint32_t *>(a.dst[c])[j] = ((const uint32_t *)s)[i];
  else static_cast<uint8_t *>(a.dst[c])[j] = ((const uint8_t *)s)[i];
}

hipError_t stage_send_reversed(const Send *seg, int n, int64_t count, hipStream_t st) {
  size_t each = 0;  // bytes of one element of every array
  for (int k = 0; k < n; k++) each += (size_t)seg[k].width;
  const size_t pad = (size_t)16 * n;
  Lease l((size_t)count * each + pad);
  if (!l.b) {  // no pinned memory to be had: reversed copies, one array at a time
    std::unique_ptr<char[]> rev(new (std::nothrow) char[(size_t)count * 8]);
    if (!rev) return hipErrorOutOfMemory;
    for (int k = 0; k < n; k++) {
      const size_t w = (size_t)seg[k].width;
      for (int64_t i = 0; i < count; i++)
        memcpy(rev.get() + i * w, static_cast<const char *>(seg[k].src) + (count - 1 - i) * w, w);
      const hipError_t e = hipMemcpyAsync(seg[k].dst, rev.get(), (size_t)count * w,
                                          hipMemcpyHostToDevice, st);
      if (e != hipSuccess) return e;
      const hipError_t e2 = hipStreamSynchronize(st);
      if (e2 != hipSuccess) return e2;
    }
    return hipSuccess;
  }
  const int64_t most = (int64_t)((l.b->bytes - pad) / each);
  for (int64_t i0 = 0; i0 < count; i0 += most) {
    SendArgs a;
    a.src = static_cast<const char *>(l.dev);
    a.count = (int)std::min(most, count - i0);
    size_t at = 0;
    for (int k = 0; k < n; k++) {
      const size_t w = (size_t)seg[k].width, bytes = (size_t)a.count * w;
      memcpy(l.b->buf + at, static_cast<const char *>(seg[k].src) + (size_t)i0 * w, bytes);
      a.dst[k] = static_cast<char *>(seg[k].dst) + (size_t)(count - i0 - a.count) * w;
      a.at[k] = (uint32_t)at;
      a.width[k] = seg[k].width;
      at += (bytes + 15) / 16 * 16;
    }
    hipLaunchKernelGGL(k_send_reversed, dim3((unsigned)((a.count + 255) / 256), (unsigned)n),
                       dim3(256), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

static int copy_threads(size_t bytes) {
  cpu_set_t set;
  CPU_ZERO(&set);
  int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
  return (int)std::max<size_t>(1, std::min<size_t>({8, (size_t)cpus, 1 + bytes / kStagePiece}));
}

hipError_t stage_fetch(const Fetch *seg, int n, hipStream_t st) {
  size_t total = 0, padded = 0;
  for (int k = 0; k < n; k++) total += seg[k].bytes, padded += (seg[k].bytes + 15) / 16 * 16;
  if (total == 0) return hipStreamSynchronize(st);
  Lease l(padded);
  if (!l.b) {  // no pinned memory to be had: straight into the arrays
    for (int k = 0; k < n; k++) {
      const hipError_t e =
          hipMemcpyAsync(seg[k].dst, seg[k].src, seg[k].bytes, hipMemcpyDeviceToHost, st);
      if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(st);
  }
  char *const buf = l.b->buf;
  const size_t bytes = l.b->bytes;
  hipEvent_t *const ev = l.b->ev;
  Piece *const window = l.b->window;
  int k = 0;
  size_t off = 0;
  while (k < n) {
    size_t at = 0, pieces = 0;
    int slice = 0;
    hipError_t r = hipSuccess;
    while (k < n && at < bytes && slice < kStageSlices && r == hipSuccess) {
      PackArgs a;
      a.dst = static_cast<char *>(l.dev);
      int np = 0;
      size_t in_slice = 0, most = 0;
      while (k < n && at < bytes && np < kFetchMax && in_slice < kStageSlice) {
        const size_t take = std::min({seg[k].bytes - off, kStagePiece, bytes - at});
        if (take) {
          a.src[np] = static_cast<const char *>(seg[k].src) + off;
          a.bytes[np] = (uint32_t)take;
          a.at[np] = (uint32_t)at;
          np++;
          window[pieces++] = {static_cast<char *>(seg[k].dst) + off, at, take, slice};
        }
        at += (take + 15) / 16 * 16;
        off += take;
        in_slice += take;
        most = std::max(most, take);
        if (off == seg[k].bytes) {
          k++;
          off = 0;
        }
      }
      if (np == 0) break;
      const unsigned gx = (unsigned)std::max<size_t>(1, std::min<size_t>(32, most / 8192));
      hipLaunchKernelGGL(k_pack, dim3(gx, (unsigned)np), dim3(256), 0, st, a);
      r = hipGetLastError();
      if (total > kStageSmall && r == hipSuccess) {
        if (l.b->nev == slice) {
          r = hipEventCreateWithFlags(&ev[slice], hipEventDisableTiming);
          if (r == hipSuccess) l.b->nev++;
        }
        if (r == hipSuccess) r = hipEventRecord(ev[slice], st);
      }
      slice++;
    }
    if (r != hipSuccess) {
      (void)hipStreamSynchronize(st);
      return r;
    }
    if (total <= kStageSmall) {
      r = hipStreamSynchronize(st);
      if (r != hipSuccess) return r;
      for (size_t q = 0; q < pieces; q++) memcpy(window[q].dst, buf + window[q].at, window[q].bytes);
      continue;  // (a great many short arrays take further windows)
    }
    std::atomic<size_t> next{0};
    std::atomic<int> bad{(int)hipSuccess};
    int device = 0;
    (void)hipGetDevice(&device);
    auto work = [&]() {
      (void)hipSetDevice(device);
      for (size_t q; (q = next.fetch_add(1)) < pieces;) {
        const hipError_t w = hipEventSynchronize(ev[window[q].slice]);
        if (w != hipSuccess) {
          bad = (int)w;
          return;
        }
        memcpy(window[q].dst, buf + window[q].at, window[q].bytes);
      }
    };
    std::thread pool[8];
    const int nt = copy_threads(at);
    for (int t = 1; t < nt; t++) {
      try {
        pool[t] = std::thread(work);
      } catch (const std::exception &) {
        break;  // no thread (or memory for one) to be had: the others take its pieces
      }
    }
    work();
    for (auto &t : pool)
      if (t.joinable()) t.join();
    if (bad != (int)hipSuccess) {
      (void)hipStreamSynchronize(st);
      return (hipError_t)bad.load();
    }
  }
  return hipSuccess;
}

}  // namespace nb

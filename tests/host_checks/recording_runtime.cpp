// The HIP runtime as the library's host code sees it, without a device. Kernels are registered by name, and a launch is
// noted; of all kernels only the copies between pinned and device memory are carried out (host_copy.hip), in order with
// the others, on one thread that stands for the stream. Device memory is what hipMalloc returned, and every address below
// 2^42, which no host allocation has; there is one gfx950 part with 256 compute units.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>

#include "uk_internal.h"

namespace {
std::mutex g_mutex;  // of the two maps
std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> m;
  return m;
}
std::map<const uint8_t*, size_t>& device_memory() {
  static std::map<const uint8_t*, size_t> m;
  return m;
}
thread_local std::string tl_kernel;
thread_local unsigned tl_grid = 0, tl_block = 0;
thread_local size_t tl_lds = 0;
thread_local int tl_launches = 0;
std::atomic<int> g_kernel_ms{0};                            // what a kernel that is not carried out takes
std::atomic<long long> g_pinned_bytes{0}, g_events{0};      // alive

struct Stream {
  std::mutex mutex;
  std::condition_variable changed;
  std::deque<std::function<void()>> tasks;
  unsigned long long enqueued = 0, done = 0;
  std::thread thread;

  unsigned long long enqueue(std::function<void()> task) {
    std::lock_guard<std::mutex> lock(mutex);
    if (!thread.joinable()) thread = std::thread([this] { work(); });
    tasks.push_back(std::move(task));
    changed.notify_all();
    return ++enqueued;
  }
  void wait(unsigned long long until) {
    std::unique_lock<std::mutex> lock(mutex);
    changed.wait(lock, [&] { return done >= until; });
  }
  void work() {
    for (;;) {
      std::function<void()> task;
      {
        std::unique_lock<std::mutex> lock(mutex);
        changed.wait(lock, [&] { return !tasks.empty(); });
        task = std::move(tasks.front());
        tasks.pop_front();
      }
      task();
      std::lock_guard<std::mutex> lock(mutex);
      ++done;
      changed.notify_all();
    }
  }
};
Stream& stream() {
  static Stream* s = new Stream();  // (its thread ends with the process)
  return *s;
}

// The arguments of the copy kernels.
struct UploadArgs {
  const uint8_t* src;
  uint8_t* dst;
  int32_t vecs;
};
struct DownloadArgs {
  const uint8_t* src;
  uint8_t* dst;
  uint32_t* flags;
  uint32_t generation;
  int32_t vecs, pieces;
};
}  // namespace

extern "C" {

// What the calling thread launched last, and how often since `recorded_reset`.
const char* recorded_kernel() { return tl_kernel.c_str(); }
unsigned recorded_grid() { return tl_grid; }
unsigned recorded_block() { return tl_block; }
size_t recorded_lds() { return tl_lds; }
int recorded_launches() { return tl_launches; }
void recorded_reset() {
  tl_kernel.clear();
  tl_launches = 0;
}
void recorded_set_kernel_ms(int ms) { g_kernel_ms = ms; }
long long recorded_pinned_bytes() { return g_pinned_bytes; }
long long recorded_events() { return g_events; }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  std::lock_guard<std::mutex> lock(g_mutex);
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }

hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t) {
  std::string name;
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    name = kernels()[host];
  }
  if (name.find("upload_kernel") != std::string::npos) {
    const UploadArgs a = *(const UploadArgs*)args[0];
    stream().enqueue([a] { memcpy(a.dst, a.src, (size_t)a.vecs * 16); });
    return hipSuccess;
  }
  if (name.find("download_kernel") != std::string::npos) {
    const DownloadArgs a = *(const DownloadArgs*)args[0];
    stream().enqueue([a] {
      const size_t bytes = (size_t)a.vecs * 16;
      for (int32_t i = 0; i < a.pieces; ++i) {
        const size_t from = (size_t)i * uk::kDownloadPieceBytes, left = bytes - from;
        memcpy(a.dst + from, a.src + from, left < (size_t)uk::kDownloadPieceBytes ? left : (size_t)uk::kDownloadPieceBytes);
        __atomic_store_n(a.flags + i, a.generation, __ATOMIC_RELEASE);
      }
    });
    return hipSuccess;
  }
  tl_kernel = name;
  tl_grid = grid.x;
  tl_block = block.x;
  tl_lds = lds;
  ++tl_launches;
  if (const int ms = g_kernel_ms) stream().enqueue([ms] { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); });
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  memset(a, 0, sizeof *a);
  bool device = (uintptr_t)p < ((uintptr_t)1 << 42);
  if (!device) {
    std::lock_guard<std::mutex> lock(g_mutex);
    auto after = device_memory().upper_bound((const uint8_t*)p);
    if (after != device_memory().begin()) {
      --after;
      device = (const uint8_t*)p < after->first + after->second;
    }
  }
  a->type = device ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
  return device ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = malloc(n);
  std::lock_guard<std::mutex> lock(g_mutex);
  device_memory()[(const uint8_t*)*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    device_memory().erase((const uint8_t*)p);
  }
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  uint8_t* block = (uint8_t*)aligned_alloc(4096, (n + 8191) / 4096 * 4096);
  *(size_t*)block = n;
  *p = block + 4096;
  g_pinned_bytes += (long long)n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  uint8_t* block = (uint8_t*)p - 4096;
  g_pinned_bytes -= (long long)*(size_t*)block;
  free(block);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipErrorInvalidValue; }
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipErrorInvalidValue; }
hipError_t hipStreamSynchronize(hipStream_t) {
  stream().wait(stream().enqueue([] {}));
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) {
  std::lock_guard<std::mutex> lock(stream().mutex);
  return stream().done == stream().enqueued ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)calloc(1, sizeof(unsigned long long));
  ++g_events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  free(e);
  --g_events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  *(unsigned long long*)e = stream().enqueue([] {});
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  stream().wait(*(unsigned long long*)e);
  return hipSuccess;
}
}

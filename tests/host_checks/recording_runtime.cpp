// The HIP runtime as the library's host code sees it, without a device: kernels are registered by name, and a launch is
// noted instead of carried out. Every pointer counts as device memory of one gfx950 part with 256 compute units.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex g_mutex;
std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> m;
  return m;
}
thread_local std::string tl_kernel;
thread_local unsigned tl_grid = 0, tl_block = 0;
thread_local size_t tl_lds = 0;
thread_local int tl_launches = 0;
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

hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3 block, void**, size_t lds, hipStream_t) {
  std::lock_guard<std::mutex> lock(g_mutex);
  tl_kernel = kernels()[host];
  tl_grid = grid.x;
  tl_block = block.x;
  tl_lds = lds;
  ++tl_launches;
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
  a->type = hipMemoryTypeDevice;
  a->devicePointer = const_cast<void*>(p);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}

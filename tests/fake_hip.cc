// fake_hip.cc -- a stand-in for the HIP runtime, preloaded by tests of the library's host code on a
// machine without a GPU: one "gfx950" device whose memory is host memory, launches that call a hook
// instead of running.  Freed memory is remembered, so a test can tell a launch that is passed a
// pointer into it.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>
#include <string>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

namespace {
std::mutex mu;
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
std::map<uintptr_t, size_t> live, freed;
typedef void (*hook_t)(const char* kernel, uint32_t grid, uint32_t block, void** args);
hook_t hook = nullptr;
struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local Config config;
char symbol[64 << 20];  // stands for every __device__ variable

bool inside(const std::map<uintptr_t, size_t>& m, uintptr_t p) {
  auto it = m.upper_bound(p);
  if (it == m.begin()) return false;
  --it;
  return p < it->first + it->second;
}
}  // namespace

extern "C" {
void fake_hip_hook(hook_t h) { hook = h; }
// Calls `each` with the name of every kernel of the libraries loaded.
void fake_hip_kernels(void (*each)(const char*)) {
  for (const auto& k : names()) each(k.second.c_str());
}
int fake_hip_freed(uint64_t p) {
  std::lock_guard<std::mutex> lock(mu);
  return inside(freed, (uintptr_t)p) && !inside(live, (uintptr_t)p);
}

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  config = {grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  if (hook) hook(names()[f].c_str(), grid.x, block.x, args);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = symbol, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = aligned_alloc(256, (n + 255) / 256 * 256);
  std::lock_guard<std::mutex> lock(mu);
  live[(uintptr_t)*p] = n;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {  // the memory itself is kept
  std::lock_guard<std::mutex> lock(mu);
  auto it = live.find((uintptr_t)p);
  if (it != live.end()) {
    freed[it->first] = it->second;
    live.erase(it);
  }
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetD16Async(hipDeviceptr_t d, unsigned short v, size_t n, hipStream_t) {
  for (size_t i = 0; i < n; ++i) static_cast<uint16_t*>(d)[i] = v;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
}

// hip_sim.cpp — the HIP runtime calls of libinferox.so, in host memory: device
// memory of a set size (allocations past it fail as on a full device), copies as
// memcpy, kernel launches counted by name and not run, no stream capture. Loaded
// before the library with global symbols, it takes the runtime's place, and the
// library's host code runs without a device.
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex mu;
std::map<void*, size_t> allocs;
size_t used = 0, limit = (size_t)8 << 30;
std::map<const void*, std::string> kernels;  // host function -> name
std::map<std::string, long> launches;
thread_local hipError_t last = hipSuccess;
hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
hipError_t take(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  if (used + n > limit) return ret(hipErrorOutOfMemory);
  *p = calloc(n ? n : 1, 1);
  allocs[*p] = n;
  used += n;
  return hipSuccess;
}
hipError_t give(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  if (!p) return hipSuccess;
  auto it = allocs.find(p);
  if (it == allocs.end()) return ret(hipErrorInvalidValue);
  used -= it->second;
  allocs.erase(it);
  free(p);
  return hipSuccess;
}
}  // namespace

extern "C" {
// ---- for the tests ----
size_t sim_used() { return used; }
void sim_limit(size_t n) { limit = n; }
long sim_launches(const char* part) {  // of the kernels whose name holds `part`
  long n = 0;
  for (auto& k : launches)
    if (k.first.find(part) != std::string::npos) n += k.second;
  return n;
}

// ---- the runtime ----
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = *b = dim3(1);
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  launches[kernels[f]]++;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char area[64 << 20]; *p = area; return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(p); }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  for (size_t i = 0; i < h; i++) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)calloc(1, 8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)calloc(1, 8); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
}

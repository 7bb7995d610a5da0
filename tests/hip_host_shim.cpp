// hip_host_shim.cpp -- the HIP runtime calls of libperman_hip.so's single
// matrix paths as host functions: device memory is host memory, kernels are
// not run, and one call can be made to fail.  Loaded before the library with
// its symbols global (tests/test_cpu_runtime_calls.py), so the library's host
// code runs without a GPU.  Test infrastructure only.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <string>

namespace {
std::string g_log;   // names of the calls, each followed by a space
std::string g_fail;  // the call that fails ...
int g_after = 0;     // ... after so many that succeed, once

hipError_t called(const char* name) {
  g_log += name;
  g_log += ' ';
  if (g_fail != name || g_after-- > 0) return hipSuccess;
  g_fail.clear();
  return hipErrorOutOfMemory;
}
template <class T>
hipError_t object(const char* name, T* out) {
  if (hipError_t e = called(name); e != hipSuccess) return e;
  *out = (T)std::calloc(1, 64);
  return hipSuccess;
}
hipError_t memory(const char* name, void** out, size_t bytes) {
  if (hipError_t e = called(name); e != hipSuccess) return e;
  *out = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
  std::memset(*out, 0, bytes);
  return hipSuccess;
}
}  // namespace

#undef hipEventCreate
extern "C" {
const char* shim_log() { return g_log.c_str(); }
void shim_clear() { g_log.clear(); }
void shim_fail(const char* name, int after) {
  g_fail = name;
  g_after = after;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "shim"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return object("hipStreamCreateWithFlags", s);
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free((void*)s);
  return called("hipStreamDestroy");
}
hipError_t hipStreamSynchronize(hipStream_t) { return called("hipStreamSynchronize"); }
hipError_t hipEventCreate(hipEvent_t* e) { return object("hipEventCreate", e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void*)e);
  return called("hipEventDestroy");
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return called("hipEventRecord"); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return called("hipEventElapsedTime");
}
hipError_t hipMalloc(void** p, size_t bytes) { return memory("hipMalloc", p, bytes); }
hipError_t hipFree(void* p) {
  std::free(p);
  return called("hipFree");
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  return memory("hipHostMalloc", p, bytes);
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return called("hipHostFree");
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::memcpy(dst, src, bytes);
  return called("hipMemcpyAsync");
}
// (around every <<<>>>: the stub between them passes the values on)
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
  *grid = *block = dim3(1, 1, 1);
  *lds = 0;
  *stream = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  return called("hipLaunchKernel");
}
}

// Host stand-in for the few HIP calls of gn_copy.h: copies happen at once, and
// the call that a test names fails.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#define __device__
#define __forceinline__ inline
#define __shared__
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum { hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
typedef void* hipStream_t;
typedef struct Event* hipEvent_t;
struct FailAt {  // the nth call from now fails (0: none)
  std::atomic<long> left{0};
  bool hit() { return left.load() > 0 && left.fetch_sub(1) == 1; }
};
inline FailAt fail_copy, fail_wait, fail_device;
inline const char* hipGetErrorString(hipError_t) { return "injected"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return fail_device.hit() ? hipErrorUnknown : hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) {
  return fail_wait.hit() ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (fail_copy.hit()) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
// device helpers of gn_common.h, never called here
struct Idx { int x; };
inline Idx threadIdx, blockDim;
template <class T> T __shfl_xor(T v, int, int) { return v; }
inline void __syncthreads() {}
#define __builtin_amdgcn_update_dpp(...) 0
inline float fmaxf(float a, float b) { return a > b ? a : b; }
inline float tanhf(float x) { return x; }

// A host-only runtime for tests without a device: copies are memcpy, done at
// once; `hipStubFailCopy` makes a copy of that number fail.
#pragma once

#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
using hipStream_t = void*;
using hipEvent_t = void*;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

inline std::atomic<int> hipStubFailCopy{-1};
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (hipStubFailCopy >= 0 && hipStubFailCopy-- == 0) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  static char event;
  *e = &event;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}

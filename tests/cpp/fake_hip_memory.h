// The rest of the fake HIP runtime: device memory, timed events and failures on
// demand (fake::fail_malloc, fake::fail_memcpy: the call that many calls from
// now fails; 0: none does).
#pragma once

#include "fake_hip.h"

namespace fake {

inline int fail_malloc = 0, fail_memcpy = 0;
inline bool fails(int& countdown) { return countdown > 0 && --countdown == 0; }
inline double clock_ms = 0;                         // advanced by the fake kernels
inline std::map<hipEvent_t, double> event_ms;

}  // namespace fake

extern "C" {

hipError_t hipMalloc(void** p, size_t n) {
  if (fake::fails(fake::fail_malloc)) return hipErrorOutOfMemory;
  *p = std::malloc(n ? n : 1);
  std::memset(*p, 0xEE, n);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
  if (fake::fails(fake::fail_memcpy)) return hipErrorUnknown;
  std::memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = new ihipStream_t(fake::device);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete s;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  std::lock_guard<std::mutex> lock(fake::mu);
  *ms = (float)(fake::event_ms[b] - fake::event_ms[a]);
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }

}  // extern "C"

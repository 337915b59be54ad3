// hip_stubs.hpp — a HIP runtime of stubs for host checks (test infrastructure only): device and
// pinned memory are ordinary memory that is counted, streams do their work at once. Included by one
// file of a program.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>

namespace stub {

inline hipError_t last_error = hipSuccess;

struct Memory {
  std::map<void*, size_t> live;
  size_t held = 0, calls = 0, largest = 0;
  size_t limit = ~size_t(0);
  hipError_t get(void** p, size_t bytes) {
    ++calls;
    largest = std::max(largest, bytes);
    if (bytes > limit - held) return last_error = hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    live[*p] = bytes;
    held += bytes;
    return hipSuccess;
  }
  hipError_t put(void* p) {
    if (!live.count(p)) return hipErrorInvalidValue;
    held -= live[p];
    live.erase(p);
    std::free(p);
    return hipSuccess;
  }
};
inline Memory pinned, device;

}  // namespace stub

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) { return stub::pinned.get(p, bytes); }
hipError_t hipHostFree(void* p) { return stub::pinned.put(p); }
hipError_t hipMalloc(void** p, size_t bytes) { return stub::device.get(p, bytes); }
hipError_t hipFree(void* p) { return stub::device.put(p); }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = stub::last_error;
  stub::last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind) {
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
}

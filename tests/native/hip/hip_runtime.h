// What download.cpp and internal.hpp use of the HIP runtime, over host memory,
// for a CPU build of download.cpp (tests/native/download_host.cpp): copies are
// done when enqueued, pinned memory is counted, one range can be called
// registered.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
using hipStream_t = struct FakeStream*;
using hipEvent_t = struct FakeEvent*;
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocPortable = 1;

inline std::atomic<int> fake_slots{0}, fake_copies{0};
inline const char* fake_registered = nullptr;  // a destination the runtime knows

inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  return *p != nullptr ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  fake_slots += *p != nullptr ? 1 : 0;
  return *p != nullptr ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p) {
  std::free(p);
  --fake_slots;
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(to, from, n);
  ++fake_copies;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = p == fake_registered ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}

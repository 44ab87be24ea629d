// The few host calls of the HIP runtime that nlm_copy.hip makes, over ordinary memory, so that
// its logic runs on a CPU: streams are ordered by doing the work at once, device memory is
// host memory, and a test makes calls fail through the `fake` counters.
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct FakeStream {
  int device;
};
struct FakeEvent {
  int device;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

namespace fake {
inline thread_local int device = 0;
inline thread_local hipError_t last = hipSuccess;
inline std::atomic<bool> failHostMalloc{false}, failEventCreate{false};
inline std::atomic<int> areas{0}, events{0};
// a caller's pinned memory, and the copies that went there
inline const char *pinned = nullptr, *pinnedEnd = nullptr;
inline std::atomic<int> pinnedCopies{0};
// copies whose destination is `watched`; a call made from the next copy, once
inline const void* watched = nullptr;
inline std::atomic<int> watchedCopies{0};
inline std::atomic<void (*)()> onCopy{nullptr};
inline bool isPinned(const void* p) { return p >= pinned && p < pinnedEnd; }
inline hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
}  // namespace fake

inline const char* hipGetErrorString(hipError_t) { return "fake error"; }
inline hipError_t hipGetLastError() {
  const hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
inline hipError_t hipGetDevice(int* d) {
  *d = fake::device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  fake::device = d;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) {
  *d = s->device;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (fake::failHostMalloc) return fake::ret(hipErrorOutOfMemory);
  *p = std::malloc(n);
  fake::areas++;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::free(p);
  fake::areas--;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (fake::failEventCreate) return fake::ret(hipErrorOutOfMemory);
  *e = new FakeEvent{fake::device};
  fake::events++;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  fake::events--;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->device == s->device ? hipSuccess : fake::ret(hipErrorInvalidHandle);
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = fake::isPinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  if (fake::isPinned(dst)) fake::pinnedCopies++;
  if (dst == fake::watched) fake::watchedCopies++;
  if (void (*f)() = fake::onCopy.exchange(nullptr)) f();
  std::memcpy(dst, src, n);
  return hipSuccess;
}

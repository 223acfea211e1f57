// The few runtime calls of cs_transfer.h for a machine without a GPU, so that
// its staging can be checked on the host: two devices, copies done at once,
// events tied to the device that was current when they were made (recording
// one on another device's stream fails, as the runtime's do), and counts of
// what was copied directly and what through the slots.
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include <map>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t { hipMemoryType type; };

struct FakeStream { int device; };
struct FakeEvent { int device; };
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

struct FakeHip {
  int device = 0;                     // the calling thread's current device
  hipError_t last = hipSuccess;
  std::map<const char*, size_t> pin;  // live hipHostMalloc blocks
  size_t direct = 0, staged = 0;      // bytes copied with the caller's array / with a slot as the host side
  int events = 0, fail_record = 0;    // live events; fail this many hipEventRecord calls
};
inline FakeHip& fake() {
  static FakeHip f;
  return f;
}
inline bool fake_pinned(const void* p) {
  auto it = fake().pin.upper_bound((const char*)p);
  if (it == fake().pin.begin()) return false;
  --it;
  return (const char*)p < it->first + it->second;
}
inline hipError_t fake_ret(hipError_t e) {
  if (e != hipSuccess) fake().last = e;
  return e;
}
inline hipError_t hipGetLastError() {
  const hipError_t e = fake().last;
  fake().last = hipSuccess;
  return e;
}
inline hipError_t hipGetDevice(int* d) {
  *d = fake().device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  fake().device = d;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) {
  *d = s->device;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = malloc(n);
  if (!*p) return fake_ret(hipErrorOutOfMemory);
  fake().pin[(const char*)*p] = n;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  fake().pin.erase((const char*)p);
  free(p);
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = fake_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new FakeEvent{fake().device};
  ++fake().events;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  --fake().events;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (fake().fail_record > 0) {
    --fake().fail_record;
    return fake_ret(hipErrorInvalidValue);
  }
  return fake_ret(e->device == s->device ? hipSuccess : hipErrorInvalidHandle);
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
  memcpy(dst, src, n);
  // the tests pin their own arrays at a whole number of 4 KiB less 8 bytes: those are no slots
  const void* host = kind == hipMemcpyDeviceToHost ? dst : src;
  bool slot = false;
  if (fake_pinned(host)) {
    auto it = --fake().pin.upper_bound((const char*)host);
    slot = it->second % 4096 == 0;
  }
  (slot ? fake().staged : fake().direct) += n;
  return hipSuccess;
}

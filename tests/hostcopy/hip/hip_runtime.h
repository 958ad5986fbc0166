// The part of the HIP runtime that fx_hostcopy.hpp calls, on host memory: devices are numbers,
// copies happen at once, an event belongs to the device that was current when it was made and can
// be recorded on that device's streams only.
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
enum hipStreamCaptureMode { hipStreamCaptureModeRelaxed = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct fakeStream { int device; };
struct fakeEvent { int device; };
using hipStream_t = fakeStream *;
using hipEvent_t = fakeEvent *;
struct hipPointerAttribute_t { hipMemoryType type; };

namespace fake {
inline thread_local int current = 0;
inline std::atomic<int> pinned{0}, mallocs{0}, staged{0}, plain{0};  // live chunks, attempts, copies of each kind
inline std::atomic<bool> no_memory{false};
inline char *chunk_base[256];
inline std::atomic<int> chunks{0};
inline bool is_chunk(const void *p)
{
  for (int i = 0; i < chunks; i++)
    if (p == chunk_base[i]) return true;
  return false;
}
}  // namespace fake

inline hipError_t hipGetDevice(int *d) { *d = fake::current; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::current = d; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *)
{
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
  fake::mallocs++;
  *p = nullptr;
  if (fake::no_memory) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  fake::chunk_base[fake::chunks++] = static_cast<char *>(*p);
  fake::pinned++;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p)
{
  std::free(p);
  fake::pinned--;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
  *e = new fakeEvent{fake::current};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t)
{
  (fake::is_chunk(kind == hipMemcpyHostToDevice ? src : dst) ? fake::staged : fake::plain)++;
  std::memcpy(dst, src, n);
  return hipSuccess;
}

/* As much of the HIP runtime's interface as host_copy.cpp uses, on the host: two devices, one
 * stream each, copies that count as in flight until an event recorded after them or their
 * stream is waited for, and failures on request. Like the runtime, it refuses to record an
 * event on another device's stream. */
#pragma once

#include <atomic>
#include <cstddef>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };

namespace fake {
struct Stream { int device; std::vector<const void *> flying; };        // host ends of its copies
struct Event { int device; Stream *stream = nullptr; size_t upto = 0; };

inline std::mutex mutex;
inline thread_local int device = 0;
inline std::map<const char *, size_t> pinned;
inline int copies = 0, direct = 0, records = 0, fail_record = -1;       // fail the n-th record

inline bool is_pinned(const void *p)
{
  const char *c = static_cast<const char *>(p);
  auto it = pinned.upper_bound(c);
  return it != pinned.begin() && c < std::prev(it)->first + std::prev(it)->second;
}
}  // namespace fake
using hipStream_t = fake::Stream *;
using hipEvent_t = fake::Event *;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = fake::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::device = d; return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  *p = ::operator new(n);
  fake::pinned[static_cast<char *>(*p)] = n;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  fake::pinned.erase(static_cast<char *>(p));
  ::operator delete(p);
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  a->type = fake::is_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
  *e = new fake::Event{fake::device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t s)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  const void *host = kind == hipMemcpyHostToDevice ? src : dst;
  std::memcpy(dst, src, n);
  ++fake::copies;
  s->flying.push_back(host);
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  if (fake::records++ == fake::fail_record) return hipErrorOutOfMemory;
  if (e->device != s->device) return hipErrorInvalidHandle;
  e->stream = s;
  e->upto = s->flying.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  // what was enqueued before the record has landed; the rest stays in flight
  if (e->stream) for (size_t k = 0; k < e->upto && k < e->stream->flying.size(); ++k) e->stream->flying[k] = nullptr;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
  std::lock_guard<std::mutex> l(fake::mutex);
  s->flying.clear();
  return hipSuccess;
}

/* Copies between host buffers and the device.
 *
 * The runtime's own copy of a pageable buffer is one thread's: 28-31 GB/s to the device (36 from
 * a buffer used just before), 18 GB/s back, and 10.5 GB/s back into a freshly allocated array, whose
 * pages that thread also has to fault in. A snapshot of a 256^3 grid (1.15 GB) so cost 40 ms in
 * and 110 ms out, four double-precision steps. Here several threads each take chunks of the
 * buffer in turn, copy them to or from two pinned slots of their own and leave the transfer of
 * one slot to run while they copy the other: 39 GB/s each way, in a new array too (256^3: 29
 * and 30 ms). The rule, by what was measured on both sides (GB/s, runtime | staged; six buffers in turn to the device,
 * a new array each time back):
 *   to the device    2 MB 22 | 15, 8 MB 26 | 22, 15 MB 28 | 26, 22 MB 28 | 31, 154 MB 31 | 38
 *   to the host      2 MB 15 | 18, 8 MB 18 | 24, 30 MB 18 | 37, 41 MB 10.5 | 30, 154 MB 10.6 | 37
 *   pinned memory    37 (2 MB) to 56 (154 MB) by the runtime, which transfers it as it is
 *
 * The staging is one per device, at most 8 threads x 2 slots x 2 MB, slots allocated when a
 * copy first needs them and freed with the last context. One copy at a time uses it: a
 * concurrent one (another host thread) takes the runtime's path instead, as do small copies.
 */
#include "host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace maragpu_host {
namespace {

constexpr size_t kChunk = size_t(2) << 20;      // a slot
// below these, the runtime's copy (staging 1.1 MB each way a step made a march through the verbs
// 12 % slower)
constexpr size_t kSmallToDevice = size_t(20) << 20, kSmallToHost = size_t(2) << 20;
constexpr size_t kPerThread = size_t(8) << 20;  // bytes that make a further thread worth its start
constexpr int kThreads = 8;
constexpr int kDevices = 64;

struct Slot {
  char *p = nullptr;
  hipEvent_t done = nullptr;
  bool ready() const { return p && done; }
  bool make()
  {
    if (ready()) return true;
    if (!p && hipHostMalloc(reinterpret_cast<void **>(&p), kChunk, hipHostMallocDefault) != hipSuccess) p = nullptr;
    if (!done && hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) done = nullptr;
    if (!ready()) (void)hipGetLastError();    // the caller has another path
    return ready();
  }
  void drop()
  {
    if (p) hipHostFree(p);
    if (done) hipEventDestroy(done);
    p = nullptr;
    done = nullptr;
  }
};

struct Staging {
  std::mutex busy;             // held by the copy that uses the slots
  int users = 0;               // guarded by g_users
  Slot slot[2 * kThreads];
};

std::mutex g_users;
Staging g_staging[kDevices];

/* The chunks of one copy, taken in turn by its threads */
struct Job {
  int device;
  hipStream_t stream;
  char *dev, *host;
  size_t n, chunk;
  bool to_device;
  std::atomic<size_t> next{0};
  std::atomic<int> error{hipSuccess};

  bool take(size_t &off, size_t &len)
  {
    if (error.load() != hipSuccess) return false;
    off = next.fetch_add(1) * chunk;
    if (off >= n) return false;
    len = std::min(chunk, n - off);
    return true;
  }
  bool ok(hipError_t e)
  {
    if (e != hipSuccess) error.store(e);
    return e == hipSuccess;
  }
  bool send(Slot &s, size_t off, size_t len)
  {
    if (!ok(to_device ? hipMemcpyAsync(dev + off, s.p, len, hipMemcpyHostToDevice, stream)
                      : hipMemcpyAsync(s.p, dev + off, len, hipMemcpyDeviceToHost, stream)))
      return false;
    if (ok(hipEventRecord(s.done, stream))) return true;
    (void)hipStreamSynchronize(stream);       // the slot is in use and has no event to wait for
    return false;
  }

  /* one thread's share, with the slots s[0], s[1]; both are idle again on return */
  void work(Slot *s)
  {
    bool flying[2] = {false, false};
    size_t off[2], len[2];
    if (to_device) {
      for (int k = 0;; k ^= 1) {
        if (flying[k] && !ok(hipEventSynchronize(s[k].done))) break;
        flying[k] = false;
        if (!take(off[k], len[k])) break;
        std::memcpy(s[k].p, host + off[k], len[k]);
        if (!send(s[k], off[k], len[k])) break;
        flying[k] = true;
      }
    }
    else {
      for (int k = 0; k < 2; ++k) flying[k] = take(off[k], len[k]) && send(s[k], off[k], len[k]);
      for (int k = 0; flying[k]; k ^= 1) {
        flying[k] = false;
        if (!ok(hipEventSynchronize(s[k].done))) break;
        std::memcpy(host + off[k], s[k].p, len[k]);
        flying[k] = take(off[k], len[k]) && send(s[k], off[k], len[k]);
      }
    }
    for (int k = 0; k < 2; ++k)
      if (flying[k]) ok(hipEventSynchronize(s[k].done));
  }
};

/* Memory that the device reads and writes as it is */
bool pinned(const void *p)
{
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeHost;
  (void)hipGetLastError();                    // a pointer the runtime does not know
  return false;
}

/* The device made current, and the caller's again afterwards: an event belongs to the device
 * that is current when it is created */
struct OnDevice {
  int before = -1;
  explicit OnDevice(int device)
  {
    if (hipGetDevice(&before) != hipSuccess || before == device || hipSetDevice(device) != hipSuccess) before = -1;
  }
  ~OnDevice() { if (before >= 0) (void)hipSetDevice(before); }
};

hipError_t copy(int device, hipStream_t stream, void *dev, void *host, size_t n, bool to_device)
{
  const OnDevice on(device);
  std::unique_lock<std::mutex> lock;
  Staging *st = device >= 0 && device < kDevices ? &g_staging[device] : nullptr;
  if (st && n >= (to_device ? kSmallToDevice : kSmallToHost) && !pinned(host))
    lock = std::unique_lock<std::mutex>(st->busy, std::try_to_lock);
  if (!lock.owns_lock() || !st->slot[0].make() || !st->slot[1].make()) {
    if (to_device) return hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, stream);
    const hipError_t e = hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }
  Job job;
  job.device = device;
  job.stream = stream;
  job.dev = static_cast<char *>(dev);
  job.host = static_cast<char *>(host);
  job.n = n;
  job.to_device = to_device;
  // a short copy in four chunks at least, so that copying and transfer overlap
  job.chunk = std::min(kChunk, (n / 4 + 4095) / 4096 * 4096);
  const unsigned cpus = std::max(1u, std::thread::hardware_concurrency() / 2);
  const size_t want = std::min<size_t>({n / kPerThread, (size_t)kThreads, (size_t)cpus});
  std::vector<std::thread> more;
  try {
    for (size_t t = 1; t < want; ++t) {
      Slot *s = &st->slot[2 * t];
      if (!s[0].make() || !s[1].make()) break;
      more.emplace_back([&job, s] {
        if (job.ok(hipSetDevice(job.device))) job.work(s);
      });
    }
  }
  catch (...) {
    // no more threads to be had: those that run share the work
  }
  job.work(&st->slot[0]);
  for (std::thread &t : more) t.join();
  return static_cast<hipError_t>(job.error.load());
}

}  // namespace

void staging_retain(int device)
{
  if (device < 0 || device >= kDevices) return;
  std::lock_guard<std::mutex> lock(g_users);
  ++g_staging[device].users;
}

void staging_release(int device)
{
  if (device < 0 || device >= kDevices) return;
  std::lock_guard<std::mutex> lock(g_users);
  Staging &st = g_staging[device];
  if (--st.users > 0) return;
  std::lock_guard<std::mutex> idle(st.busy);
  for (Slot &s : st.slot) s.drop();
}

hipError_t copy_to_device(int device, hipStream_t stream, void *dev, const void *host, size_t n)
{
  return copy(device, stream, dev, const_cast<void *>(host), n, true);
}

hipError_t copy_to_host(int device, hipStream_t stream, void *host, const void *dev, size_t n)
{
  return copy(device, stream, const_cast<void *>(dev), host, n, false);
}

}  // namespace maragpu_host

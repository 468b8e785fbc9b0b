/* host_copy.cpp on the stand-in runtime (tests/host/runtime): one copy, and what it left. */
#include "../../ctf_amd/csrc/host_copy.cpp"

extern "C" {

/* Copies n bytes between `host` and a "device" buffer on device `device` from a thread whose
 * current device is `current`; out: the result, copies made, copies still in flight, the
 * thread's device afterwards. pinned: `host` is memory of the runtime's. */
void run_copy(int device, int current, int to_device, char *host, char *dev, size_t n, int pinned, int fail_record,
              int *out)
{
  fake::Stream stream{device, {}};
  fake::device = current;
  fake::copies = fake::records = 0;
  fake::fail_record = fail_record;
  if (pinned) fake::pinned[host] = n;
  maragpu_host::staging_retain(device);
  const hipError_t e = to_device ? maragpu_host::copy_to_device(device, &stream, dev, host, n)
                                 : maragpu_host::copy_to_host(device, &stream, host, dev, n);
  out[0] = e;
  out[1] = fake::copies;
  out[2] = 0;
  for (const void *p : stream.flying) out[2] += p && p != host;      // the caller waits for its own buffer
  out[3] = fake::device;
  maragpu_host::staging_release(device);
  if (pinned) fake::pinned.erase(host);
}

}

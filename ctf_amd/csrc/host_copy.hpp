/* Copies between host buffers and the device, large pageable ones through pinned staging
 * (host_copy.cpp). */
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace maragpu_host {

/* Every context holds a reference to its device's staging; the last one to go frees it. */
void staging_retain(int device);
void staging_release(int device);

/* n bytes from host to dev, or from dev to host, in order with the work already on `stream`
 * (of `device`, which has a context; another device may be current). copy_to_host returns with the bytes in
 * place; after copy_to_device the caller synchronises the stream before the host buffer
 * changes hands, as after hipMemcpyAsync. */
hipError_t copy_to_device(int device, hipStream_t stream, void *dev, const void *host, size_t n);
hipError_t copy_to_host(int device, hipStream_t stream, void *host, const void *dev, size_t n);

}  // namespace maragpu_host

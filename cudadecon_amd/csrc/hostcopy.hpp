// Copies between caller-owned (pageable) host buffers and the device.
//
// Measured on an MI355X host for 1 GiB: pageable hipMemcpy 26 GB/s to the
// device and 17 GB/s back, pinned 57 GB/s both ways, one host thread's
// memcpy 29 GB/s.  Copies of some size therefore go through pinned staging
// buffers: the DMA of one chunk overlaps several host threads copying another
// chunk between the caller's memory and its pinned buffer.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace cdn {

// host -> device, after the work already queued on `st`.  Returns once the
// data is on the device.
void copy_to_device(hipStream_t st, void* dev, const void* host, size_t bytes);

// device -> host, after the work already queued on `st`.  Returns once the
// data is in the host buffer.  fresh_stream: `st` was made for this call.
void copy_to_host(hipStream_t st, void* host, const void* dev, size_t bytes, bool fresh_stream = false);

}  // namespace cdn

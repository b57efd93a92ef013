// Copies between the caller's (pageable) host arrays and the device through a
// pinned ring, with the host side of the copy spread over a few threads.
//
// The runtime copies pageable memory with one thread: 18 GB/s from the device
// and 38 GB/s to it on an MI355X host whose link does 57 GB/s; a 16.8 MB
// image took 960 us of an 8.2 ms render, and a denoiser inference of 0.6 ms of
// kernels took 3 ms. Here each chunk's transfer overlaps the other chunks' host
// copies.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace mdwt {

// Kernels and host threads take turns on a ring's slots, each after the other's
// event: the memory is coherent and the events release to the system, and the
// protocol needs both. A lane is one ring with its events and threads; a device has
// at most four.
//
// A handle that copies holds a reference while it lives; the lanes are given back with
// the last one.
void host_copy_acquire();
void host_copy_release();

// dst (host) = src (device); returns when dst is complete. Ordered after the
// work already on s.
hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t s);
// dst (device) = src (host). Later work on s sees dst; src may be read until s has
// been synchronized (small arrays: they go to the runtime's own copy, and waiting for
// it cost a denoiser inference of 16^2 to 128^2 pixels 8 us of 190).
hipError_t copy_to_device(void* dst, const void* src, size_t bytes, int device, hipStream_t s);

}  // namespace mdwt

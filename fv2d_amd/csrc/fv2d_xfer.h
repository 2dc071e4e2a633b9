// fv2d_xfer.h -- copies between pageable host arrays and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

namespace fv2d {

// Copies `bytes` between a pageable host array and device memory, in the order of stream `st` of
// device `dev` (the calling thread's current device); return when the copy is done.
hipError_t copy_to_host(void *dst, const void *dev_src, size_t bytes, int dev, hipStream_t st);
hipError_t copy_to_device(void *dev_dst, const void *src, size_t bytes, int dev, hipStream_t st);

// Every handle and batch on a device holds a reference to the device's pinned buffers; the last
// release gives them back.
void copy_retain(int dev);
void copy_release(int dev);

}  // namespace fv2d

// Large device-to-host reads of field data into pageable (numpy) memory.
#pragma once

#include <cstddef>

#include <hip/hip_runtime.h>

namespace mpa {

// Copies bytes from device to host after the work queued on s, and waits.
void read_back(void* host, const void* dev, size_t bytes, hipStream_t s);

// Worlds alive in the process: the last one to go gives read_back's pinned
// buffers back to the system, unless they were read through since there was no
// world (a world per point of a sweep keeps them).
void readback_retain();
void readback_release();

}  // namespace mpa

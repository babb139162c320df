// Large device-to-host reads of field data into pageable (numpy) memory.
#pragma once

#include <cstddef>

#include <hip/hip_runtime.h>

namespace mpa {

// Copies bytes from device to host after the work queued on s, and waits.
void read_back(void* host, const void* dev, size_t bytes, hipStream_t s);

// Worlds alive in the process: the pinned buffers of read_back go back to the
// system with the last one.
void readback_retain();
void readback_release();

}  // namespace mpa

// Device-to-host copies of results into the caller's memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace lbm {

struct HostCopy {
  void* dst;        // caller's memory
  const void* src;  // device memory
  size_t bytes;
};

// Copies the parts after the work queued on `stream`, and returns when they have arrived.
hipError_t read_back(const HostCopy* parts, int n, hipStream_t stream);

// Solver objects hold the staging memory of read_back while they live: it is allocated by the first
// copy that needs it and freed with the last object.
void readout_hold();
void readout_release();

}  // namespace lbm

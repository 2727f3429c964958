// vrh_copy.h -- device to host copies of large results.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

// Pinned staging of one handle (8 MB, made on the first large copy, freed
// with the handle).  Not shared: a handle is used by one thread at a time.
struct HostCopy {
  static constexpr int kSlots = 8;
  char *pin = nullptr;
  hipEvent_t ev[kSlots] = {};
};
// dst[0, bytes) = src after the work on st; complete on return.
hipError_t host_download(HostCopy &c, hipStream_t st, void *dst, const void *src, size_t bytes);
void host_copy_free(HostCopy &c);

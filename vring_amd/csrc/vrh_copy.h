// vrh_copy.h -- device to host copies of large results.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

// Pinned staging of one handle (8 MB, made on the first large copy, freed
// with the handle), used by one large copy at a time: threads that fetch
// results of the same handle take turns.
struct HostCopy {
  static constexpr int kSlots = 8;
  std::mutex mu;
  char *pin = nullptr;
  hipEvent_t ev[kSlots] = {};
};
// dst[0, bytes) = src after the work on st; complete on return.
hipError_t host_download(HostCopy &c, hipStream_t st, void *dst, const void *src, size_t bytes);
void host_copy_free(HostCopy &c);

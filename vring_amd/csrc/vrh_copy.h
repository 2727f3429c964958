// vrh_copy.h -- device to host copies of large results.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

// Staging of one handle's large results, made once it pays and freed with the
// handle: pinned slots (8 MB), and on the device a buffer of the largest result
// so far, in which particle rows and the pressure solve's array stand as well.
// One call uses them at a time: threads that fetch results of the same handle
// take turns.
struct HostCopy {
  static constexpr int kSlots = 8;
  std::recursive_mutex mu;
  size_t fetched = 0;           // bytes of large results so far
  char *pin = nullptr;
  hipEvent_t ev[kSlots] = {};
  hipStream_t st = nullptr;     // of the copies into the slots
  hipEvent_t taken = nullptr;   // the result is complete and out of the way of later work
  char *dev = nullptr;
  size_t cap = 0;
};
// dst[0, bytes) = src at this point of st; complete on return.  own: no other
// thread queues work that writes src while the call runs.
hipError_t host_download(HostCopy &c, hipStream_t st, void *dst, const void *src, size_t bytes, bool own = false);
// c.dev holds at least `bytes` (false: no memory).  Its user keeps c.mu locked.
bool host_room(HostCopy &c, size_t bytes);
void host_copy_free(HostCopy &c);

// vrh_copy.cpp -- large results from the device to a caller's host array.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "vrh_copy.h"

namespace {

// A result usually goes to fresh pageable memory, where the runtime's copy is
// bound by one thread that takes the page faults and copies out of its own
// staging memory (11 GB/s for 48 MB, 16 for 17 MB; the link carries 55).  Four
// threads that each copy out of pinned slots of their own, two chunks on their
// way, took a 48 MB particle download from 5.1 to 2.1 ms and one of 17 MB from
// 1.17 to 0.87; chunks of 512 KB 2.8 ms, of 2 MB 1.9 with twice the pinned
// memory, eight threads 2.2.  Below 8 MB the gain (0.33 -> 0.28 ms at 4 MB)
// would not pay for the pinned memory.  That takes 1 to 1.2 ms once: less than a
// result of 32 MB gains (35 MB: 3.5 -> 1.4 ms), but more than a few of 9 or 17 MB
// do (0.1 and 0.3 ms each), so for these it is made once the handle has fetched
// 64 MB.  Uploads gain nothing (0.61 ms for 17 MB either way).
constexpr size_t kChunk = (size_t)1 << 20;
constexpr int kThreads = 4, kDepth = 2;
constexpr size_t kMin = (size_t)8 << 20, kAtOnce = (size_t)32 << 20, kPays = (size_t)64 << 20;

struct Job {
  HostCopy *c;
  int dev;
  char *dst;
  const char *src;
  size_t bytes;
  std::atomic<size_t> next{0};
  std::atomic<hipError_t> err{hipSuccess};  // the first failure
  bool ok(hipError_t e) {
    hipError_t none = hipSuccess;
    if (e != hipSuccess) err.compare_exchange_strong(none, e);
    return e == hipSuccess;
  }
};

// Takes chunks from the job's counter until none is left, keeping kDepth of
// them on their way into its own slots while it copies the oldest out.
void worker(Job *b, int q) {
  if (!b->ok(hipSetDevice(b->dev))) return;
  const size_t nc = (b->bytes + kChunk - 1) / kChunk;
  size_t id[kDepth];
  auto len = [&](size_t c) { return std::min(kChunk, b->bytes - c * kChunk); };
  auto issue = [&](int s) {
    id[s] = b->next.fetch_add(1);
    if (id[s] >= nc) return;
    const int g = q * kDepth + s;
    if (!b->ok(hipMemcpyAsync(b->c->pin + g * kChunk, b->src + id[s] * kChunk, len(id[s]), hipMemcpyDeviceToHost,
                              b->c->st)) ||
        !b->ok(hipEventRecord(b->c->ev[g], b->c->st)))
      id[s] = nc;
  };
  for (int s = 0; s < kDepth; s++) issue(s);
  for (int s = 0; id[s] < nc; s = (s + 1) % kDepth) {
    const int g = q * kDepth + s;
    if (!b->ok(hipEventSynchronize(b->c->ev[g]))) return;
    memcpy(b->dst + id[s] * kChunk, b->c->pin + g * kChunk, len(id[s]));
    issue(s);
  }
}

bool ready(HostCopy &c) {
  if (c.pin) return true;
  auto event = [](hipEvent_t &e) {
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) e = nullptr;
    return e != nullptr;
  };
  bool ok = event(c.taken);
  for (hipEvent_t &e : c.ev) ok = ok && event(e);
  if (ok && !c.st && hipStreamCreateWithFlags(&c.st, hipStreamNonBlocking) != hipSuccess) c.st = nullptr;
  ok = ok && c.st;
  if (ok && hipHostMalloc((void **)&c.pin, HostCopy::kSlots * kChunk, hipHostMallocDefault) != hipSuccess) c.pin = nullptr;
  if (!c.pin) (void)hipGetLastError();
  return c.pin != nullptr;
}

}  // namespace

static_assert(kThreads * kDepth == HostCopy::kSlots, "one slot for every chunk on its way");

bool host_room(HostCopy &c, size_t bytes) {
  if (c.cap >= bytes) return true;
  if (c.dev) (void)hipFree(c.dev);
  c.dev = nullptr;
  c.cap = 0;
  if (hipMalloc((void **)&c.dev, bytes) != hipSuccess) {
    c.dev = nullptr;
    (void)hipGetLastError();
    return false;
  }
  c.cap = bytes;
  return true;
}

hipError_t host_download(HostCopy &c, hipStream_t st, void *dst, const void *src, size_t bytes, bool own) {
  // memory that the runtime knows (pinned, managed) takes the copy engine's
  // writes directly
  hipPointerAttribute_t at{};
  const bool known = hipPointerGetAttributes(&at, dst) == hipSuccess && at.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  // the stream's device is current while its events and copies are made
  int dev = 0, cur = 0;
  bool staged = bytes >= kMin && !known && hipStreamGetDevice(st, &dev) == hipSuccess && hipGetDevice(&cur) == hipSuccess;
  struct Back {
    int dev;
    bool on;
    ~Back() { if (on) (void)hipSetDevice(dev); }
  } back{cur, staged && cur != dev};
  if (back.on) staged = hipSetDevice(dev) == hipSuccess;
  std::unique_lock<std::recursive_mutex> turn(c.mu, std::defer_lock);
  if (staged) {
    turn.lock();
    if (c.fetched < kPays) c.fetched += bytes;
    staged = c.pin || bytes >= kAtOnce || c.fetched >= kPays;
  }
  if (!staged || !ready(c) || !(own || host_room(c, bytes))) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }
  // The chunks leave one after another, and work that another thread queues on
  // st meanwhile could write src between two of them: they come from a copy
  // that is taken in one piece, on a stream of their own (17 MB: 873 us; 877
  // straight from src).
  hipError_t e = hipSuccess;
  if (!own) {
    e = hipMemcpyAsync(c.dev, src, bytes, hipMemcpyDeviceToDevice, st);
    src = c.dev;
  }
  if (e == hipSuccess) e = hipEventRecord(c.taken, st);
  if (e == hipSuccess) e = hipStreamWaitEvent(c.st, c.taken, 0);
  if (e != hipSuccess) return e;
  Job b;
  b.c = &c;
  b.dev = dev;
  b.dst = static_cast<char *>(dst);
  b.src = static_cast<const char *>(src);
  b.bytes = bytes;
  std::thread th[kThreads - 1];
  try {
    for (int q = 1; q < kThreads; q++) th[q - 1] = std::thread(worker, &b, q);
  } catch (const std::exception &) {  // no more threads or no memory for one: the others take its chunks
  }
  worker(&b, 0);
  for (std::thread &t : th)
    if (t.joinable()) t.join();
  (void)b.ok(hipStreamSynchronize(c.st));
  return b.err;
}

void host_copy_free(HostCopy &c) {
  if (c.st) (void)hipStreamDestroy(c.st);
  if (c.pin) (void)hipHostFree(c.pin);
  if (c.dev) (void)hipFree(c.dev);
  if (c.taken) (void)hipEventDestroy(c.taken);
  for (hipEvent_t &e : c.ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  c.st = nullptr;
  c.pin = c.dev = nullptr;
  c.taken = nullptr;
  c.cap = 0;
}

// A test double of the HIP runtime calls that libvrh makes, loaded before the
// runtime (LD_PRELOAD) so that the library's host code runs without a GPU.
// "Device" memory is host memory; copies, fills and events are real and in
// stream order, each stream with a thread of its own; a kernel launch does
// nothing but is counted by name, with its LDS and with a cost on its
// stream's clock, which events read.  Calls can be made to fail by count.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

using Op = std::function<void()>;

struct Stream {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<Op> q;
  size_t put = 0, ran = 0;
  bool stop = false;
  double clock = 0.0;  // touched by the stream's own thread only
  std::thread th{[this] {
    for (;;) {
      Op op;
      {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [this] { return stop || !q.empty(); });
        if (q.empty()) return;
        op = std::move(q.front());
        q.pop_front();
      }
      op();
      std::lock_guard<std::mutex> l(mu);
      ran++;
      cv.notify_all();
    }
  }};
  void push(Op op) {
    std::lock_guard<std::mutex> l(mu);
    q.push_back(std::move(op));
    put++;
    cv.notify_all();
  }
  void drain() {
    std::unique_lock<std::mutex> l(mu);
    const size_t n = put;
    cv.wait(l, [&] { return ran >= n; });
  }
  ~Stream() {
    { std::lock_guard<std::mutex> l(mu); stop = true; cv.notify_all(); }
    th.join();
  }
};
struct Event {
  std::mutex mu;
  std::condition_variable cv;
  size_t recorded = 0, done = 0;
  double t = 0.0;
  void wait(size_t n) {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return done >= n; });
  }
};
struct Graph { std::vector<std::function<void(Stream *)>> ops; };
struct Kern { long runs = 0, lds = 0; const void *ptr = nullptr; };

std::mutex g_mu;
std::map<const void *, std::string> g_names;
std::map<const void *, long> g_granted;
std::map<std::string, Kern> g_kern;
std::map<const char *, size_t> g_live;    // device allocations
std::map<const char *, size_t> g_pinned;  // pinned host allocations
long g_graphs = 0, g_dead = 0, g_refused = 0;
bool g_lds_refused = false;
std::atomic<long> g_fail_malloc{0}, g_fail_copy{0};  // 1: the next call fails; n: the n-th; -1: all
thread_local hipError_t t_err = hipSuccess;
thread_local Graph *t_cap = nullptr;
thread_local struct { dim3 grid, block; size_t lds; hipStream_t st; } t_cfg;

hipError_t err(hipError_t e) { return t_err = e; }
bool fails(std::atomic<long> &n) {
  const long v = n.load();
  if (v < 0) return true;
  return v > 0 && n.fetch_sub(1) == 1;
}
Stream *str(hipStream_t s) {
  static Stream *null = new Stream;
  return s ? reinterpret_cast<Stream *>(s) : null;
}
void enqueue(hipStream_t s, std::function<void(Stream *)> f) {
  if (t_cap) { t_cap->ops.push_back(std::move(f)); return; }
  Stream *q = str(s);
  q->push([q, f = std::move(f)] { f(q); });
}
bool inside(const std::map<const char *, size_t> &m, const void *p) {
  std::lock_guard<std::mutex> l(g_mu);
  auto it = m.upper_bound(static_cast<const char *>(p));
  if (it == m.begin()) return false;
  --it;
  return static_cast<const char *>(p) < it->first + it->second;
}

}  // namespace

#define API extern "C" __attribute__((visibility("default")))

// ---- controls ----
API void dbl_reset() { std::lock_guard<std::mutex> l(g_mu); g_kern.clear(); g_graphs = g_dead = g_refused = 0; }
API void dbl_fail(long mallocs, long copies) { g_fail_malloc = mallocs; g_fail_copy = copies; }
API void dbl_refuse_lds(int on) { g_lds_refused = on != 0; }
// launches run since the reset of kernels whose name holds `part`, their
// largest LDS, and what else was counted
API long dbl_runs(const char *part) {
  std::lock_guard<std::mutex> l(g_mu);
  long n = 0;
  for (auto &k : g_kern) if (k.first.find(part) != std::string::npos) n += k.second.runs;
  return n;
}
API long dbl_lds(const char *part) {
  std::lock_guard<std::mutex> l(g_mu);
  long n = 0;
  for (auto &k : g_kern) if (k.first.find(part) != std::string::npos && k.second.lds > n) n = k.second.lds;
  return n;
}
// what the last launch of such a kernel was given (see hipLaunchKernel)
API const void *dbl_given(const char *part) {
  std::lock_guard<std::mutex> l(g_mu);
  for (auto &k : g_kern) if (k.first.find(part) != std::string::npos) return k.second.ptr;
  return nullptr;
}
API long dbl_graphs() { return g_graphs; }    // graphs instantiated
API long dbl_dead() { return g_dead; }        // launches that were given freed memory
API long dbl_refused() { return g_refused; }  // launches refused
API long dbl_pinned() {                       // bytes of pinned memory
  std::lock_guard<std::mutex> l(g_mu);
  long n = 0;
  for (auto &a : g_pinned) n += (long)a.second;
  return n;
}

// ---- devices ----
API hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
API hipError_t hipSetDevice(int) { return hipSuccess; }
API hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
API hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { *d = 0; return hipSuccess; }
API int hipGetStreamDeviceId(hipStream_t) { return 0; }
API hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 163840; return hipSuccess; }
API hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v) {
  if (g_lds_refused) return err(hipErrorInvalidValue);
  std::lock_guard<std::mutex> l(g_mu);
  g_granted[f] = v;
  return hipSuccess;
}
API hipError_t hipGetLastError() { const hipError_t e = t_err; t_err = hipSuccess; return e; }
API const char *hipGetErrorString(hipError_t e) {
  thread_local std::string s;
  s = "error " + std::to_string((int)e);
  return s.c_str();
}
API hipError_t hipGetSymbolAddress(void **p, const void *) { static char scratch[1 << 20]; *p = scratch; return hipSuccess; }

// ---- memory ----
API hipError_t hipMalloc(void **p, size_t n) {
  if (fails(g_fail_malloc)) { *p = nullptr; return err(hipErrorOutOfMemory); }
  char *m = static_cast<char *>(std::calloc(n ? n : 1, 1));
  std::lock_guard<std::mutex> l(g_mu);
  g_live[m] = n;
  *p = m;
  return hipSuccess;
}
// freed memory is only forgotten, so that a use of it can be seen and does no harm
API hipError_t hipFree(void *p) { std::lock_guard<std::mutex> l(g_mu); g_live.erase(static_cast<char *>(p)); return hipSuccess; }
API hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  char *m = static_cast<char *>(std::calloc(n, 1));
  std::lock_guard<std::mutex> l(g_mu);
  g_pinned[m] = n;
  *p = m;
  return hipSuccess;
}
API hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> l(g_mu);
  g_pinned.erase(static_cast<char *>(p));
  std::free(p);
  return hipSuccess;
}
API hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  *a = hipPointerAttribute_t{};
  a->type = inside(g_pinned, p) ? hipMemoryTypeHost : inside(g_live, p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
  return hipSuccess;
}
API hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t s) {
  if (fails(g_fail_copy)) return err(hipErrorInvalidValue);
  if (kind == hipMemcpyHostToDevice && !inside(g_pinned, src)) {  // pageable: taken before the call returns
    auto tmp = std::make_shared<std::vector<char>>(static_cast<const char *>(src), static_cast<const char *>(src) + n);
    enqueue(s, [=](Stream *) { std::memcpy(dst, tmp->data(), n); });
    return hipSuccess;
  }
  enqueue(s, [=](Stream *) {
    // a large copy over the link takes its time
    if (kind == hipMemcpyDeviceToHost && n >= 65536) std::this_thread::sleep_for(std::chrono::microseconds(n >> 12));
    std::memcpy(dst, src, n);
  });
  if (kind == hipMemcpyDeviceToHost && !inside(g_pinned, dst) && !t_cap) str(s)->drain();
  return hipSuccess;
}
API hipError_t hipMemsetAsync(void *dst, int v, size_t n, hipStream_t s) {
  enqueue(s, [=](Stream *) { std::memset(dst, v, n); });
  return hipSuccess;
}

// ---- streams and events ----
API hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(new Stream); return hipSuccess; }
API hipError_t hipStreamDestroy(hipStream_t s) { str(s)->drain(); delete str(s); return hipSuccess; }
API hipError_t hipStreamSynchronize(hipStream_t s) { str(s)->drain(); return hipSuccess; }
API hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new Event); return hipSuccess; }
API hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
API hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); return hipSuccess; }
API hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (t_cap) return hipSuccess;  // a captured step's operations stay in their order
  Event *v = reinterpret_cast<Event *>(e);
  size_t n;
  { std::lock_guard<std::mutex> l(v->mu); n = ++v->recorded; }
  enqueue(s, [=](Stream *q) {
    std::lock_guard<std::mutex> l(v->mu);
    if (n > v->done) { v->done = n; v->t = q->clock; }
    v->cv.notify_all();
  });
  return hipSuccess;
}
API hipError_t hipEventSynchronize(hipEvent_t e) {
  Event *v = reinterpret_cast<Event *>(e);
  size_t n;
  { std::lock_guard<std::mutex> l(v->mu); n = v->recorded; }
  v->wait(n);
  return hipSuccess;
}
API hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (t_cap) return hipSuccess;
  Event *v = reinterpret_cast<Event *>(e);
  size_t n;
  { std::lock_guard<std::mutex> l(v->mu); n = v->recorded; }
  enqueue(s, [=](Stream *q) {
    v->wait(n);
    std::lock_guard<std::mutex> l(v->mu);
    q->clock = (v->t > q->clock ? v->t : q->clock) + 5.0;
  });
  return hipSuccess;
}
API hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(1e-3 * (reinterpret_cast<Event *>(b)->t - reinterpret_cast<Event *>(a)->t));
  return hipSuccess;
}

// ---- graphs ----
API hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { t_cap = new Graph; return hipSuccess; }
API hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = reinterpret_cast<hipGraph_t>(t_cap); t_cap = nullptr; return hipSuccess; }
API hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *x = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(g)));
  std::lock_guard<std::mutex> l(g_mu);
  g_graphs++;
  return hipSuccess;
}
API hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  Graph g = *reinterpret_cast<Graph *>(x);
  enqueue(s, [g](Stream *q) { for (auto &o : g.ops) o(q); });
  return hipSuccess;
}
API hipError_t hipGraphDestroy(hipGraph_t g) { delete reinterpret_cast<Graph *>(g); return hipSuccess; }
API hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete reinterpret_cast<Graph *>(x); return hipSuccess; }

// ---- kernels ----
API void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
API void __hipUnregisterFatBinary(void **) {}
API void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
API void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
  std::lock_guard<std::mutex> l(g_mu);
  g_names[host] = name;
}
API hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { t_cfg = {g, b, lds, s}; return hipSuccess; }
API hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = t_cfg.grid; *b = t_cfg.block; *lds = t_cfg.lds; *s = t_cfg.st;
  return hipSuccess;
}
API hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t s) {
  std::string name;
  {
    std::lock_guard<std::mutex> l(g_mu);
    name = g_names[f];
    const long limit = g_granted.count(f) ? g_granted[f] : 65536;
    if ((long)lds > limit || !grid.x || !grid.y || !grid.z || block.x * block.y * block.z > 1024) {
      g_refused++;
      return err(hipErrorInvalidValue);
    }
  }
  // the matrix of a dense z transform (first member of its fourth argument)
  // and the axial metric of the projection (of its third)
  const bool zd = name.find("k_zdense") != std::string::npos && name.find("k_zdense2") == std::string::npos;
  const void *ptr = zd ? *static_cast<const void **>(args[3])
                    : name.find("k_project") != std::string::npos ? *static_cast<const void **>(args[2]) : nullptr;
  enqueue(s, [=](Stream *q) {
    const bool dead = ptr && !inside(g_live, ptr);
    std::lock_guard<std::mutex> l(g_mu);
    Kern &k = g_kern[name];
    k.runs++;
    if ((long)lds > k.lds) k.lds = (long)lds;
    k.ptr = ptr;
    g_dead += dead;
    q->clock += 10.0;
  });
  return hipSuccess;
}

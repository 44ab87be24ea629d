// nlm_copy.hip -- copies between the device and a caller's ordinary (pageable) memory.
//
// hipMemcpy to pageable memory goes through the runtime's own staging, one thread
// filling the destination: 17.8 GB/s measured for 128 MB, and less into freshly
// allocated pages, against 56.8 GB/s into pinned memory.  Here large results run through a
// pinned staging area in 1 MB pieces, two per participant in flight, and the caller and up to
// three helper threads move the pieces to the destination.  That pays from about 3 MB (a
// batch's result of 6.2 MB 816 -> 766 us for the call, 12.5 MB 2.24 -> 1.35 ms, two of 16 MB 2.02 ->
// 1.28; at 2 MB 50 us slower), and for one caller at a time: callers that come meanwhile take the
// runtime's copy, since several at once are bound by the transfers (four threads with two
// results of 16.8 MB each: 3.23 ms a pass, 3.22 all by the runtime, 3.93 by way of the area).
// Small results are gathered in the area and share one wait; between the two the runtime's own
// copy is used, as for every upload, whose source pages are there already (in pieces by the helpers a 6.2 MB input made the call 766 -> 1395 us).
// Calls, ms before -> now: Chi2PDC Green's N = 512 (C, S of 4 MB each) 2.63 -> 2.37, N =
// 32 0.116 -> 0.080; Chi3 z-grids N = 512, nZ = 1000 (48 MB) 11.4 -> 10.6.
#include <sched.h>
#include <sys/types.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "../../include/nlm.h"
#include "nlm_copy.hpp"

namespace {

constexpr size_t PIECE = (size_t)1 << 20;
constexpr size_t LARGE = 3 * PIECE;        // through the pieces
constexpr size_t SMALL = (size_t)256 << 10;  // gathered in the staging area
constexpr int HELPERS = 3, PARTS = HELPERS + 1, SLOTS = 2 * PARTS;
// with fewer the helpers take turns with the caller: results of 4.2 MB, two a call, 0.62 ms on one
// CPU and 0.50 on two against 0.48 by the runtime's copies, 0.47 on three, 0.42 on four
constexpr int MIN_CPUS = 3;
constexpr int MAX_IDLE = 4;  // staging areas kept per process between copies (8 MB each)

struct Staging {
  int device = 0;
  char* buf = nullptr;
  hipEvent_t ev[SLOTS] = {};
  char* slot(int k) { return buf + (size_t)k * PIECE; }
  void destroy() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (buf) (void)hipHostFree(buf);
    delete this;
  }
};

// Staging areas: taken for the length of one copy, so concurrent callers never share
// one; at most MAX_IDLE are kept, the others are freed when they come back.
std::mutex g_mu;
Staging* g_idle[MAX_IDLE];
int g_idles = 0;

// Of the stream's device, whichever is current: an event is recorded on its own device only.
hipError_t take(hipStream_t stream, Staging** out) {
  int dev = 0, cur = 0;
  hipError_t e = hipStreamGetDevice(stream, &dev);
  if (e == hipSuccess) e = hipGetDevice(&cur);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (int k = 0; k < g_idles; k++)
      if (g_idle[k]->device == dev) {
        *out = g_idle[k];
        g_idle[k] = g_idle[--g_idles];
        return hipSuccess;
      }
  }
  Staging* s = new (std::nothrow) Staging();
  if (!s) return hipErrorOutOfMemory;
  s->device = dev;
  if (cur != dev) e = hipSetDevice(dev);
  if (e == hipSuccess) e = hipHostMalloc((void**)&s->buf, SLOTS * PIECE, hipHostMallocDefault);
  for (int k = 0; k < SLOTS && e == hipSuccess; k++) e = hipEventCreateWithFlags(&s->ev[k], hipEventDisableTiming);
  if (cur != dev) (void)hipSetDevice(cur);
  if (e != hipSuccess) {
    s->destroy();
    return e;
  }
  *out = s;
  return hipSuccess;
}

void give(Staging* s) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_idles < MAX_IDLE) {
      g_idle[g_idles++] = s;
      return;
    }
  }
  s->destroy();
}

// Work for the caller and the helpers: part 0..PARTS-1 of it on each.
struct Job {
  virtual void run(int part) = 0;
};

// Helper threads, started at the first large copy and kept for the process.  One copy
// uses them at a time; another that comes meanwhile does without.
class Helpers {
 public:
  // every part of the job; false if the helpers are busy
  bool run(Job& job) {
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (!use.owns_lock() || !start()) return false;
    {
      std::lock_guard<std::mutex> lk(mu_);
      job_ = &job;
      left_ = HELPERS;
      round_++;
    }
    go_.notify_all();
    job.run(0);
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [&] { return left_ == 0; });
    job_ = nullptr;
    return true;
  }

 private:
  bool start() {
    if (started_ > 0 && pid_ != getpid()) return false;  // a forked child has none of its parent's threads
    pid_ = getpid();
    // each part once: helpers that could not be started are started by a later copy
    try {
      for (; started_ < HELPERS; started_++) std::thread([this, k = started_ + 1] { loop(k); }).detach();
    } catch (...) {
      return false;
    }
    return true;
  }
  void loop(int part) {
    unsigned long seen = 0;
    for (;;) {
      Job* job;
      {
        std::unique_lock<std::mutex> lk(mu_);
        go_.wait(lk, [&] { return round_ != seen; });
        seen = round_;
        job = job_;
      }
      job->run(part);
      {
        std::lock_guard<std::mutex> lk(mu_);
        left_--;
      }
      done_.notify_one();
    }
  }
  std::mutex use_, mu_;
  std::condition_variable go_, done_;
  Job* job_ = nullptr;
  int left_ = 0;
  unsigned long round_ = 0;
  int started_ = 0;
  pid_t pid_ = 0;
};

Helpers& helpers() {
  static Helpers* h = new Helpers();  // never destroyed: its threads outlive main
  return *h;
}

// One participant's share of a large copy: pieces part, part + parts, ..., alternating
// between its two slots.
hipError_t share(Staging* st, char* host, const char* dev, size_t bytes, int part, int parts, hipStream_t s) {
  const size_t n = (bytes + PIECE - 1) / PIECE;
  const auto len = [&](size_t c) { return std::min(PIECE, bytes - c * PIECE); };
  hipError_t e = hipSuccess;
  size_t pending[2] = {n, n};
  size_t c = (size_t)part;
  int k = 0;
  for (; c < n + 2 * (size_t)parts && e == hipSuccess; c += (size_t)parts, k ^= 1) {
    const int q = 2 * part + k;
    if (pending[k] < n) {  // the piece this slot still holds
      e = hipEventSynchronize(st->ev[q]);
      if (e != hipSuccess) break;
      memcpy(host + pending[k] * PIECE, st->slot(q), len(pending[k]));
      pending[k] = n;
    }
    if (c >= n) continue;
    e = hipMemcpyAsync(st->slot(q), dev + c * PIECE, len(c), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(st->ev[q], s);
    pending[k] = c;
  }
  return e;
}

// CPUs that this thread, and helpers started by it, may run on
int cpus() {
  cpu_set_t set;
  return sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : PARTS;
}

std::atomic<int> g_large{0};  // large copies under way in the process

hipError_t large(Staging* st, char* host, const char* dev, size_t bytes, hipStream_t s) {
  struct Shares : Job {
    Staging* st;
    char* host;
    const char* dev;
    size_t bytes;
    hipStream_t s;
    hipError_t errs[PARTS] = {};
    void run(int part) override {
      if (part > 0) {
        errs[part] = hipSetDevice(st->device);
        if (errs[part] != hipSuccess) return;
      }
      errs[part] = share(st, host, dev, bytes, part, PARTS, s);
    }
  } job;
  job.st = st;
  job.host = host;
  job.dev = dev;
  job.bytes = bytes;
  job.s = s;
  struct Entered {
    const int others = g_large.fetch_add(1);
    ~Entered() { g_large.fetch_sub(1); }
  } entered;
  if (entered.others > 0 || cpus() < MIN_CPUS || !helpers().run(job))
    return hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
  for (hipError_t e : job.errs)
    if (e != hipSuccess) return e;
  return hipSuccess;
}

// Whether the runtime knows the memory (pinned, managed, a device's): its own copy then goes
// there directly.  Two results of 67 MB into pinned arrays 4.32 -> 2.37 ms.
bool known(const void* host) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

// Without a staging area (no pinned memory left): the runtime's own copies.
hipError_t plain(const HostCopy* items, int n, hipStream_t s) {
  hipError_t e = hipSuccess;
  for (int i = 0; i < n && e == hipSuccess; i++)
    if (items[i].host && items[i].bytes)
      e = hipMemcpyAsync(items[i].host, items[i].dev, items[i].bytes, hipMemcpyDeviceToHost, s);
  const hipError_t w = hipStreamSynchronize(s);
  return e == hipSuccess ? w : e;
}

int failed(hipError_t e) {
  return set_err(NLM_DEVICE_ERROR, std::string("HIP error in a copy: ") + hipGetErrorString(e));
}

}  // namespace

int nlm_to_host(const HostCopy* items, int n, hipStream_t s) {
  Staging* st = nullptr;
  hipError_t e = take(s, &st);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    e = plain(items, n, s);
    return e == hipSuccess ? NLM_OK : failed(e);
  }
  size_t at = 0;
  int first = 0;
  // small items are gathered in the staging area and waited for together
  const auto flush = [&](int end) {
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    size_t o = 0;
    for (int i = first; i < end && e == hipSuccess; i++) {
      if (!items[i].host || items[i].bytes == 0 || items[i].bytes > SMALL || known(items[i].host)) continue;
      memcpy(items[i].host, st->buf + o, items[i].bytes);
      o += items[i].bytes;
    }
    first = end;
    at = 0;
  };
  for (int i = 0; i < n && e == hipSuccess; i++) {
    const HostCopy& c = items[i];
    if (!c.host || c.bytes == 0) continue;
    if (known(c.host)) {
      e = hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, s);
    } else if (c.bytes >= LARGE) {
      flush(i);
      first = i + 1;
      if (e == hipSuccess) e = large(st, (char*)c.host, (const char*)c.dev, c.bytes, s);
    } else if (c.bytes > SMALL) {
      e = hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, s);
    } else {
      if (at + c.bytes > SLOTS * PIECE) flush(i);
      if (e == hipSuccess) e = hipMemcpyAsync(st->buf + at, c.dev, c.bytes, hipMemcpyDeviceToHost, s);
      at += c.bytes;
    }
  }
  if (e == hipSuccess) flush(n);
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(s);  // nothing may still write the area
    st->destroy();
    return failed(e);
  }
  give(st);
  return NLM_OK;
}

int nlm_to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
  if (bytes == 0) return NLM_OK;
  const hipError_t e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
  return e == hipSuccess ? NLM_OK : failed(e);
}

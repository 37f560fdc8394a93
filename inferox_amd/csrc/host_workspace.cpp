// host_workspace.cpp — device workspaces kept between operator calls
// (host_workspace.h).
#include "host_workspace.h"

namespace ifx {

namespace {

struct Idle {
  void* p;
  size_t bytes;
  int dev;
};
// fixed arrays: nothing here may throw across the C boundary
struct IdleList {
  Idle v[kLeaseSlots + 1];
  int n = 0;
  Idle remove(int i) {
    const Idle x = v[i];
    for (int j = i + 1; j < n; j++) v[j - 1] = v[j];
    n--;
    return x;
  }
};
std::mutex g_mu;
IdleList g_idle;  // oldest first

std::mutex g_stream_mu;
void* g_stream_ws = nullptr;
size_t g_stream_bytes = 0;
hipStream_t g_stream_of = nullptr;  // the stream it was allocated on

size_t round_up(size_t b) { return (b + (1 << 20) - 1) >> 20 << 20; }

bool free_idle() {
  IdleList v;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    v = g_idle;
    g_idle.n = 0;
  }
  for (int i = 0; i < v.n; i++) (void)hipFree(v.v[i].p);
  return v.n > 0;
}

// (g_stream_mu held) the stream's workspace back to its pool, in stream order
bool free_stream() {
  const bool had = g_stream_ws;
  if (had) (void)hipFreeAsync(g_stream_ws, g_stream_of);
  g_stream_ws = nullptr;
  g_stream_bytes = 0;
  return had;
}

// (g_stream_mu held) and from the pool to the device
void drain_stream() {
  (void)hipStreamSynchronize(g_stream_of);
  hipMemPool_t pool;
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess)
    (void)hipMemPoolTrimTo(pool, 0);
}

}  // namespace

bool workspace_give_up() {
  (void)hipGetLastError();  // of the allocation that failed
  bool any = free_idle();
  std::lock_guard<std::mutex> lk(g_stream_mu);
  if (free_stream()) {
    drain_stream();
    any = true;
  }
  return any;
}

hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory && workspace_give_up()) e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the caller has the status; the next launch's is its own
    *p = nullptr;
  }
  return e;
}

hipError_t WorkspaceLease::take(size_t bytes) {
  give_back();
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  {  // the smallest idle buffer that holds it
    std::lock_guard<std::mutex> lk(g_mu);
    int best = -1;
    for (int i = 0; i < g_idle.n; i++)
      if (g_idle.v[i].dev == dev && g_idle.v[i].bytes >= bytes &&
          (best < 0 || g_idle.v[i].bytes < g_idle.v[best].bytes))
        best = i;
    if (best >= 0) {
      const Idle x = g_idle.remove(best);
      p_ = x.p;
      bytes_ = x.bytes;
      dev_ = dev;
      return hipSuccess;
    }
  }
  const size_t n = round_up(bytes);
  e = device_malloc(&p_, n);
  if (e != hipSuccess) return e;
  bytes_ = n;
  dev_ = dev;
  return hipSuccess;
}

void WorkspaceLease::give_back() {
  if (!p_) return;
  IdleList drop;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_idle.v[g_idle.n++] = Idle{p_, bytes_, dev_};  // n was at most kLeaseSlots
    size_t total = 0;
    for (int i = 0; i < g_idle.n; i++) total += g_idle.v[i].bytes;
    while (g_idle.n > kLeaseSlots || total > kLeaseKept) {
      const Idle x = g_idle.remove(0);
      total -= x.bytes;
      drop.v[drop.n++] = x;
    }
  }
  p_ = nullptr;
  for (int i = 0; i < drop.n; i++) (void)hipFree(drop.v[i].p);
}

StreamWorkspace::StreamWorkspace(hipStream_t st) : lock_(g_stream_mu), st_(st) {}

hipError_t StreamWorkspace::take(size_t bytes) {
  const bool keep = bytes <= kStreamWsKept;
  if (keep && bytes <= g_stream_bytes) {
    p_ = g_stream_ws;
    return hipSuccess;
  }
  if (keep) free_stream();
  const size_t n = keep ? round_up(bytes) : bytes;
  hipError_t e = hipMallocAsync(&p_, n, st_);
  if (e == hipErrorOutOfMemory) {  // what is kept may be what is missing
    (void)hipGetLastError();
    free_idle();
    free_stream();
    g_stream_of = st_;
    drain_stream();
    e = hipMallocAsync(&p_, n, st_);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    p_ = nullptr;
    return e;
  }
  if (keep) {
    g_stream_ws = p_;
    g_stream_bytes = n;
    g_stream_of = st_;
  } else {
    own_ = true;
  }
  return hipSuccess;
}

StreamWorkspace::~StreamWorkspace() {
  if (own_ && p_) (void)hipFreeAsync(p_, st_);
}

void workspace_trim() {
  free_idle();
  std::lock_guard<std::mutex> lk(g_stream_mu);
  free_stream();
}

}  // namespace ifx

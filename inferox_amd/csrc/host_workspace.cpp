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

size_t round_up(size_t b) { return (b + (1 << 20) - 1) >> 20 << 20; }

void free_idle() {
  IdleList v;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    v = g_idle;
    g_idle.n = 0;
  }
  for (int i = 0; i < v.n; i++) (void)hipFree(v.v[i].p);
}

}  // namespace

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
  e = hipMalloc(&p_, n);
  if (e != hipSuccess) {  // what is kept may be what is missing
    free_idle();
    (void)hipGetLastError();
    e = hipMalloc(&p_, n);
  }
  if (e != hipSuccess) {
    p_ = nullptr;
    return e;
  }
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
  if (bytes > kStreamWsKept) {
    own_ = true;
    return hipMallocAsync(&p_, bytes, st_);
  }
  if (bytes > g_stream_bytes) {
    if (g_stream_ws) (void)hipFreeAsync(g_stream_ws, st_);
    g_stream_ws = nullptr;
    g_stream_bytes = 0;
    const size_t n = round_up(bytes);
    const hipError_t e = hipMallocAsync(&g_stream_ws, n, st_);
    if (e != hipSuccess) {
      g_stream_ws = nullptr;
      return e;
    }
    g_stream_bytes = n;
  }
  p_ = g_stream_ws;
  return hipSuccess;
}

StreamWorkspace::~StreamWorkspace() {
  if (own_ && p_) (void)hipFreeAsync(p_, st_);
}

void workspace_trim(hipStream_t st) {
  free_idle();
  std::lock_guard<std::mutex> lk(g_stream_mu);
  if (g_stream_ws) (void)hipFreeAsync(g_stream_ws, st);
  g_stream_ws = nullptr;
  g_stream_bytes = 0;
}

}  // namespace ifx

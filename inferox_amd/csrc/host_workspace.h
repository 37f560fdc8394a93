// host_workspace.h — device workspaces kept between operator calls.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

namespace ifx {

// An exclusive buffer for one call that waits for its stream before it
// returns (the attention operators, a session's short prompts).  With hipMalloc and hipFree (which waits for the whole device) in
// each call a decode attention over 2048 rows took 43.6 us, 23.3 with buffers
// kept for the next call (its kernels: 9.5); over 8192 rows 94.2 and 30.3.  At
// most kLeaseSlots buffers and kLeaseKept bytes are kept over all devices; they
// go when the last uploaded matrix is freed (workspace_trim; what later calls
// leave is kept again) and when an allocation finds no memory.  A buffer
// belongs to one call at a time, so calls on several threads and streams never
// share one.
constexpr int kLeaseSlots = 8;
constexpr size_t kLeaseKept = 128ull << 20;
class WorkspaceLease {
 public:
  WorkspaceLease() = default;
  WorkspaceLease(const WorkspaceLease&) = delete;
  WorkspaceLease& operator=(const WorkspaceLease&) = delete;
  ~WorkspaceLease() { give_back(); }
  hipError_t take(size_t bytes);
  void give_back();  // every launch that uses the buffer has completed
  void* ptr() const { return p_; }

 private:
  void* p_ = nullptr;
  size_t bytes_ = 0;
  int dev_ = -1;
};

// The workspace of asynchronous calls on the library's own stream, which lives
// until the process ends: launches on it run in order, so consecutive calls
// share one buffer.  The lock is held while a call enqueues its launches (the
// launches of two threads' calls may not interleave).  Grown and freed in
// stream order; requests past kStreamWsKept are not kept.  (A stream-ordered
// allocation per call goes back to the system at every synchronisation: a
// matmul_qt of 8 rows waited for by itself took 318 us, 70 with this.)
constexpr size_t kStreamWsKept = 256ull << 20;
class StreamWorkspace {
 public:
  explicit StreamWorkspace(hipStream_t library_stream);
  ~StreamWorkspace();
  hipError_t take(size_t bytes);
  void* ptr() const { return p_; }

 private:
  std::unique_lock<std::mutex> lock_;
  hipStream_t st_;
  void* p_ = nullptr;
  bool own_ = false;  // this call's alone: freed with it
};

// Frees what is kept and not in use (called when the last uploaded matrix goes).
void workspace_trim();
// The same for an allocation that found no memory: what was kept is back with
// the device on return.  Whether there was anything.
bool workspace_give_up();
// hipMalloc that gives up what is kept before it fails; leaves no last error.
// Every device allocation of the library that outlives a call is one.
hipError_t device_malloc(void** p, size_t bytes);

}  // namespace ifx

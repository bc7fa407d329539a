// Device arrays copied out to the caller's pageable memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace kc {

// One copy of `bytes` from device memory to the caller's `dst` at the end of a
// call; bytes are whole words and src is aligned to 16 bytes.  The constructor
// (at the call's start; dst may be null: nothing to do) lets helper threads
// fault in dst's pages while the GPU works, without changing what they hold.
// enqueue() may put a small copy into the stream ahead of a wait the caller
// makes anyway (waited: that is over); finish() copies, src final in stream
// order, and returns when dst is written.  Destroying it without finish()
// leaves dst as it was.  Throws Failure.
class CopyOut {
 public:
  CopyOut(void *dst, size_t bytes, int device);
  ~CopyOut();
  CopyOut(const CopyOut &) = delete;
  CopyOut &operator=(const CopyOut &) = delete;
  void enqueue(const void *src, hipStream_t stream);
  void finish(const void *src, hipStream_t stream, bool waited = false);

 private:
  struct Job;
  Job *job_ = nullptr;     // large copies: the helpers' shared state
  char *ring_ = nullptr;   // the borrowed pinned memory
  bool queued_ = false;    // a small copy into it is in stream_
  hipStream_t stream_ = nullptr;
  void *dst_;
  size_t bytes_;
  int device_;
};

// Handles that copy out hold a reference; the pinned staging memory is given
// back with the last one.
void copy_out_retain();
void copy_out_release();

}  // namespace kc

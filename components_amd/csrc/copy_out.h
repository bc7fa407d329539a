// Results to the caller's pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace kc {

// One copy of `count` 32-bit numbers below `bound` from device memory to the
// caller's `dst` at the end of a call; src is aligned to 16 bytes.  The constructor
// (at the call's start; dst may be null: nothing to do) lets helper threads
// fault in dst's pages while the GPU works, without changing what they hold.
// enqueue() puts the first transfers into the stream, ahead of a wait the
// caller makes anyway; finish() copies, src final in stream order, and returns
// when dst is written.  Destroying it without finish() leaves dst as it was.
// Throws Failure.
class CopyOut {
 public:
  CopyOut(uint32_t *dst, size_t count, uint64_t bound);
  ~CopyOut();
  CopyOut(const CopyOut &) = delete;
  CopyOut &operator=(const CopyOut &) = delete;
  void enqueue(const uint32_t *src, hipStream_t stream);
  void finish(const uint32_t *src, hipStream_t stream);

 private:
  struct Job;
  friend struct Helpers;
  void issue();
  Job *job_ = nullptr;
  const uint32_t *src_ = nullptr;
  hipStream_t stream_ = nullptr;
  bool queued_ = false;  // transfers into the ring are in the stream
};

// Handles whose calls copy results keep the pinned ring and the helper threads
// alive; the last one gives them back.
void copy_out_retain();
void copy_out_release();

}  // namespace kc

// Labels to the caller's pageable memory.  hipMemcpy moved them through the
// runtime's staging buffer on one thread, which also took the page faults of
// a fresh buffer: 10 GB/s (16.8 M labels: 6.4 ms beside 7 to 9 ms of GPU work),
// against 56 GB/s into pinned memory.  Here a ring of pinned slots takes the
// transfers while helper threads move finished slots on, and the pages are faulted
// in while the GPU still works.
#include "copy_out.h"

#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "kc_common.h"

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace kc {

namespace {

// (short transfers leave gaps between them: 64 of 1 MB took 2.3 ms where 16 of
// 4 MB take 1.6)
constexpr size_t kSlotBytes = 4 << 20;
constexpr int kSlots = 4;
constexpr size_t kPieceBytes = 512 << 10;  // moved on by one helper
// below this one copy into pinned memory and one memcpy: a thread costs more
constexpr size_t kThreadsMin = 1 << 20;
constexpr int kMaxHelpers = 8;
constexpr size_t kFaultBytes = 2 << 20;

// The pinned ring: one for the process (16 MB, with an event per slot), lent
// to one copy at a time and given back with the last handle.
struct Ring {
  std::mutex m;
  int handles = 0;
  bool lent = false;
  char *mem = nullptr;
  int device = -1;  // the events' device
  hipEvent_t events[kSlots] = {};
} g_ring;

// (the caller holds the mutex)
void ring_drop_events() {
  for (hipEvent_t &e : g_ring.events) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  g_ring.device = -1;
}

void ring_drop() {
  ring_drop_events();
  if (g_ring.mem) (void)hipHostFree(g_ring.mem);
  g_ring.mem = nullptr;
}

// Null when another copy holds the ring or it cannot be had.
char *ring_borrow(int device) {
  std::lock_guard<std::mutex> lock(g_ring.m);
  if (g_ring.lent) return nullptr;
  if (!g_ring.mem) {
    void *p = nullptr;
    if (hipHostMalloc(&p, kSlotBytes * kSlots, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_ring.mem = static_cast<char *>(p);
  }
  if (g_ring.device != device) {
    ring_drop_events();
    for (hipEvent_t &e : g_ring.events)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        e = nullptr;
        return nullptr;
      }
    g_ring.device = device;
  }
  g_ring.lent = true;
  return g_ring.mem;
}

void ring_return() {
  std::lock_guard<std::mutex> lock(g_ring.m);
  g_ring.lent = false;
  if (g_ring.handles == 0) ring_drop();
}

// A transfer by stores from the CUs: 50 GB/s always, where the copy engine that
// hipMemcpyAsync picks runs at 57 or, for long stretches on some streams, at
// 20 (67 MB: 3.6 instead of 1.6 ms).  What bounds it is the host link; 64
// workgroups fill it (16: 5% slower).
constexpr unsigned kTransferBlocks = 64;

__global__ __launch_bounds__(kBlock) void k_transfer(uint32_t *dst, const uint32_t *src, uint64_t words) {
  const uint64_t quads = words / 4, stride = static_cast<uint64_t>(gridDim.x) * kBlock;
  const uint64_t first = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  for (uint64_t i = first; i < quads; i += stride)
    reinterpret_cast<uint4 *>(dst)[i] = reinterpret_cast<const uint4 *>(src)[i];
  if (first < words % 4) dst[4 * quads + first] = src[4 * quads + first];
}

// src and bytes: whole words, src aligned to 16 (device arrays and their
// multiples of a piece).
void transfer(void *slot, const void *src, size_t bytes, hipStream_t s) {
  hipLaunchKernelGGL(k_transfer, dim3(kTransferBlocks), dim3(kBlock), 0, s, static_cast<uint32_t *>(slot),
                     static_cast<const uint32_t *>(src), bytes / 4);
  KC_LAUNCH_CHECK();
}

// Faults in the whole pages inside [p, p + bytes) for writing (their contents
// stay); where the kernel cannot, the copy takes the faults.
void fault_in(char *p, size_t bytes) {
  const uintptr_t page = static_cast<uintptr_t>(sysconf(_SC_PAGESIZE));
  const uintptr_t a = (reinterpret_cast<uintptr_t>(p) + page - 1) / page * page;
  const uintptr_t z = (reinterpret_cast<uintptr_t>(p) + bytes) / page * page;
  if (z > a) (void)madvise(reinterpret_cast<void *>(a), z - a, MADV_POPULATE_WRITE);
}

}  // namespace

// Pages and chunks are claimed one after another by whichever helper is free,
// so the copy does not depend on how many threads there are (at least one).
struct CopyOut::Job {
  char *dst = nullptr;
  size_t bytes = 0;
  int helpers = 0;
  std::thread first;                // starts the other helpers and joins them
  std::mutex m;
  std::condition_variable changed;  // some of the following moved on
  size_t next_fault = 0;            // bytes whose pages are claimed
  // once the copy begins: transfers of `chunk` bytes, one ring slot each, moved
  // on in pieces
  size_t chunk = 0;
  size_t ready = 0;                 // bytes that have reached their slots
  size_t claimed = 0, done = 0;     // bytes taken and moved by helpers
  std::vector<size_t> left;         // per transfer: bytes still in its slot
  bool stop = false;
  const char *ring = nullptr;

  void help() {
    std::unique_lock<std::mutex> lock(m);
    while (!stop) {
      if (claimed < ready) {
        const size_t at = claimed, c = at / chunk;
        const size_t n = std::min({kPieceBytes, (c + 1) * chunk - at, bytes - at});
        claimed += n;
        lock.unlock();
        std::memcpy(dst + at, ring + (c % kSlots) * kSlotBytes + (at - c * chunk), n);
        lock.lock();
        left[c] -= n;
        done += n;
        if (left[c] == 0) changed.notify_all();
      } else if (claimed >= bytes) {
        return;
      } else if (next_fault < bytes) {
        const size_t at = next_fault;
        next_fault += kFaultBytes;
        lock.unlock();
        fault_in(dst + at, std::min(kFaultBytes, bytes - at));
        lock.lock();
      } else {
        changed.wait(lock);
      }
    }
  }
  void start() {
    first = std::thread([this] {
      std::vector<std::thread> others;
      try {
        for (int h = 1; h < helpers; ++h) others.emplace_back([this] { help(); });
      } catch (...) {  // fewer helpers then
      }
      help();
      for (auto &t : others) t.join();
    });
  }
  void end() {
    {
      std::lock_guard<std::mutex> lock(m);
      stop = true;
      changed.notify_all();
    }
    if (first.joinable()) first.join();
  }
  ~Job() { end(); }
};

CopyOut::CopyOut(void *dst, size_t bytes, int device) : dst_(dst), bytes_(dst ? bytes : 0), device_(device) {
  if (bytes_ <= kThreadsMin) return;
  std::unique_ptr<Job> j(new Job);
  j->dst = static_cast<char *>(dst);
  j->bytes = bytes;
  const int cpus = static_cast<int>(std::thread::hardware_concurrency());
  j->helpers = std::max(1, std::min({kMaxHelpers, cpus / 2, static_cast<int>(bytes_ / kThreadsMin)}));
  try {
    j->start();
  } catch (...) {  // no thread to be had: finish() copies the plain way
    return;
  }
  job_ = j.release();
}

CopyOut::~CopyOut() {
  delete job_;
  if (queued_) (void)hipStreamSynchronize(stream_);
  if (ring_) ring_return();
}

void CopyOut::enqueue(const void *src, hipStream_t stream) {
  if (!bytes_ || bytes_ > kThreadsMin) return;
  if (!ring_) ring_ = ring_borrow(device_);
  if (!ring_) return;
  transfer(ring_, src, bytes_, stream);
  queued_ = true;
  stream_ = stream;
}

void CopyOut::finish(const void *src, hipStream_t stream, bool waited) {
  if (!bytes_) return;
  if (bytes_ <= kThreadsMin) {
    waited = waited && queued_;
    if (!queued_) enqueue(src, stream);
    if (queued_) {
      if (!waited) KC_HIP(hipStreamSynchronize(stream));
      queued_ = false;
      std::memcpy(dst_, ring_, bytes_);
      return;
    }
  } else if (job_) {
    ring_ = ring_borrow(device_);
  }
  if (!ring_ || !job_) {  // another copy holds the ring, or there is no helper
    KC_HIP(hipMemcpyAsync(dst_, src, bytes_, hipMemcpyDeviceToHost, stream));
    KC_HIP(hipStreamSynchronize(stream));
    return;
  }
  Job &j = *job_;
  // short copies in at least four transfers, so that moving overlaps them
  const size_t chunk = std::min(kSlotBytes, (bytes_ / 4 + kPieceBytes - 1) / kPieceBytes * kPieceBytes);
  const size_t chunks = (bytes_ + chunk - 1) / chunk;
  {
    std::lock_guard<std::mutex> lock(j.m);
    j.chunk = chunk;
    j.left.resize(chunks);
    for (size_t c = 0; c < chunks; ++c) j.left[c] = std::min(chunk, bytes_ - c * chunk);
    j.ring = ring_;
  }
  // however this ends, the helpers stop and no copy into the ring is left in
  // the stream
  struct Drain {
    Job &j;
    hipStream_t s;
    ~Drain() {
      j.end();
      (void)hipStreamSynchronize(s);
    }
  } drain{j, stream};
  // (only this thread talks to the runtime)
  size_t issued = 0, arrived = 0;
  while (arrived < chunks) {
    while (issued < chunks && issued < arrived + kSlots) {
      if (issued >= kSlots) {  // its slot's last transfer has to be moved on first
        std::unique_lock<std::mutex> lock(j.m);
        if (j.left[issued - kSlots] != 0) {
          if (issued > arrived) break;
          j.changed.wait(lock, [&] { return j.left[issued - kSlots] == 0; });
        }
      }
      const size_t off = issued * chunk;
      transfer(ring_ + (issued % kSlots) * kSlotBytes, static_cast<const char *>(src) + off,
               std::min(chunk, bytes_ - off), stream);
      KC_HIP(hipEventRecord(g_ring.events[issued % kSlots], stream));
      ++issued;
    }
    KC_HIP(hipEventSynchronize(g_ring.events[arrived % kSlots]));
    ++arrived;
    std::lock_guard<std::mutex> lock(j.m);
    j.ready = std::min(arrived * chunk, bytes_);
    j.changed.notify_all();
  }
  std::unique_lock<std::mutex> lock(j.m);
  j.changed.wait(lock, [&] { return j.done == bytes_; });
}

void copy_out_retain() {
  std::lock_guard<std::mutex> lock(g_ring.m);
  ++g_ring.handles;
}

void copy_out_release() {
  std::lock_guard<std::mutex> lock(g_ring.m);
  if (--g_ring.handles == 0 && !g_ring.lent) ring_drop();
}

}  // namespace kc

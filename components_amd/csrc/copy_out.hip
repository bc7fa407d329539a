// Labels to the caller's pageable memory.  hipMemcpy moved them through the
// runtime's staging buffer on one thread, which also took the page faults of
// a fresh buffer: 10 GB/s (16.8 M labels: 6.4 ms beside 7 to 9 ms of GPU work),
// against 56 GB/s into pinned memory.  Here kernels store them into a pinned
// ring, helper threads move them on piece by piece as the pieces arrive, and the
// pages are faulted in while the GPU still works.
#include "copy_out.h"

#include <sched.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "kc_common.h"

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace kc {

namespace {

// The ring takes 4 M numbers: four slots, each what one transfer fills once the
// ring has been round.
constexpr size_t kSlotCount = 1 << 20;
constexpr int kSlots = 4;
constexpr size_t kRingCount = kSlots * kSlotCount, kRingBytes = 4 * kRingCount;
// what one thread moves on at once (64 k numbers take it about 28 us)
constexpr size_t kPiece = 64 << 10, kLargePiece = 128 << 10;
// Above this with helper threads.  Below, waking them takes longer, and the
// calling thread, which faults the pages in while the transfer is under way,
// moves whole words: 100 000 labels 25 us, where helpers took 48, three bytes a
// label 36, and hipMemcpy 28; 250 000 labels 45, 64, 77, 55.
constexpr size_t kHelpersMin = 256 << 10;
constexpr int kMaxHelpers = 8;
constexpr size_t kFaultBytes = 512 << 10;

// Numbers cross the link in as few bytes as the largest needs, two, three (with
// helpers) or four: output word i (8 bytes) of n packed numbers.
__device__ __forceinline__ uint64_t packed_word(int width, const uint32_t *src, uint64_t n, uint64_t i) {
  const auto at = [&](uint64_t k) -> uint64_t { return k < n ? src[k] : 0u; };
  if (width == 4) return at(2 * i) | at(2 * i + 1) << 32;
  if (width == 2) return at(4 * i) | at(4 * i + 1) << 16 | at(4 * i + 2) << 32 | at(4 * i + 3) << 48;
  const uint64_t k = 8 * i / 3;  // the number that byte 8 i belongs to, and its bytes before that one
  const int s = static_cast<int>(8 * i - 3 * k);
  uint64_t v = at(k) >> 8 * s | at(k + 1) << (24 - 8 * s) | at(k + 2) << (48 - 8 * s);
  if (s == 2) v |= at(k + 3) << 56;
  return v;
}

// A transfer by stores from the CUs: 50 GB/s always, where the copy engine that
// hipMemcpyAsync picks runs at 57 or, for long stretches on some streams, at
// 20 (67 MB: 3.6 instead of 1.6 ms).  What bounds it is the host link, so the
// numbers are packed (16.8 M at three bytes 1.29 -> 1.06 ms, 5.9 M at two 0.42
// -> 0.21); 64 workgroups fill it (16: 5% slower).
// Every workgroup tells of its share of every piece by a word of its own in
// pinned memory, so that the host needs neither an event nor a launch per piece.
constexpr unsigned kTransferBlocks = 64;

template <int kWidth>
__global__ __launch_bounds__(kBlock) void k_transfer(char *dst, const uint32_t *src, uint64_t count, uint64_t piece,
                                                     uint32_t *arrived, uint32_t value) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
  const uint64_t first = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  for (uint64_t at = 0, p = 0; at < count; at += piece, ++p) {
    const uint64_t n = min(piece, count - at), words = (n * kWidth + 7) / 8;
    uint64_t *to = reinterpret_cast<uint64_t *>(dst + at * kWidth);  // (a piece is a multiple of 8 numbers)
    for (uint64_t i = first; i < words; i += stride) host_store(to + i, packed_word(kWidth, src + at, n, i));
    host_stores_done();
    __syncthreads();
    if (threadIdx.x == 0) host_store(arrived + p * kTransferBlocks + blockIdx.x, value);
  }
}

// The host's side: n numbers of `width` bytes each to dst (which need not be
// aligned).
void unpack(char *dst, const char *src, size_t n, int width) {
  if (width == 4) {
    std::memcpy(dst, src, 4 * n);
    return;
  }
  uint32_t *to = reinterpret_cast<uint32_t *>(dst);
  if (width == 2) {
    const uint16_t *from = reinterpret_cast<const uint16_t *>(src);
    for (size_t i = 0; i < n; ++i) to[i] = from[i];
    return;
  }
  for (size_t i = 0; i < n; ++i) {  // (the last reads a byte past them, inside the ring's memory)
    uint32_t x;
    std::memcpy(&x, src + 3 * i, 4);
    to[i] = x & 0xFFFFFFu;
  }
}

constexpr size_t kArrivedBytes = kRingCount / kPiece * kTransferBlocks * sizeof(uint32_t);

// The pinned ring: one for the process (16 MB and the arrival words), lent to
// one copy at a time and given back with the last handle.
struct Ring {
  std::mutex m;
  int handles = 0;
  bool lent = false;
  char *mem = nullptr;
  uint32_t value = 0;  // of the last transfer (the borrower's)
} g_ring;

void ring_drop() {
  if (g_ring.mem) (void)hipHostFree(g_ring.mem);
  g_ring.mem = nullptr;
}

// Null when another copy holds the ring or it cannot be had.
char *ring_borrow() {
  std::lock_guard<std::mutex> lock(g_ring.m);
  if (g_ring.lent) return nullptr;
  if (!g_ring.mem) {
    void *p = nullptr;
    if (hipHostMalloc(&p, kRingBytes + kArrivedBytes, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_ring.mem = static_cast<char *>(p);
    std::memset(g_ring.mem + kRingBytes, 0, kArrivedBytes);
    g_ring.value = 0;
  }
  g_ring.lent = true;
  return g_ring.mem;
}

void ring_return() {
  std::lock_guard<std::mutex> lock(g_ring.m);
  g_ring.lent = false;
  if (g_ring.handles == 0) ring_drop();
}

// Faults in the whole pages inside [p, p + bytes) for writing (their contents
// stay); where the kernel cannot, the copy takes the faults.
void fault_in(char *p, size_t bytes) {
  const uintptr_t page = static_cast<uintptr_t>(sysconf(_SC_PAGESIZE));
  const uintptr_t a = (reinterpret_cast<uintptr_t>(p) + page - 1) / page * page;
  const uintptr_t z = (reinterpret_cast<uintptr_t>(p) + bytes) / page * page;
  if (z > a) (void)madvise(reinterpret_cast<void *>(a), z - a, MADV_POPULATE_WRITE);
}

// A spinning thread's turn: a pause, and after a while the CPU to others.
struct Spin {
  int turns = 0;
  void operator()() {
    if (++turns < 2000)
      __builtin_ia32_pause();
    else
      sched_yield();
  }
};

}  // namespace

// Pieces and pages are claimed one after another by whichever thread is free,
// so a copy does not depend on how many helpers there are, or whether any.
struct CopyOut::Job {
  char *dst = nullptr;
  size_t count = 0, bytes = 0, piece = 0, pieces = 0;  // numbers, their bytes at dst, numbers a piece, pieces
  int width = 4;                                       // bytes of a number in the ring
  unsigned blocks = 0;
  // under the helpers' mutex
  bool listed = false, hot = false;  // hot: the transfers are in the stream
  int users = 0;                     // helpers at work on it
  size_t next_fault = 0;             // bytes whose pages are claimed
  // the copy itself
  char *ring = nullptr;
  uint32_t first_value = 0;              // of the first transfer; the later ones count on
  size_t issued = 0;                     // numbers with a transfer in the stream (the calling thread's)
  std::atomic<size_t> next_piece{0};     // claimed
  std::atomic<size_t> done{0};           // numbers moved
  std::unique_ptr<std::atomic<size_t>[]> left;  // per slot's turn: numbers still in it
  std::atomic<bool> commit{false}, stop{false};

  size_t slot_turns() const { return (count + kSlotCount - 1) / kSlotCount; }
  // the transfer that a slot's turn belongs to: the first fills the whole ring
  uint32_t value_of(size_t turn) const { return first_value + static_cast<uint32_t>(turn < kSlots ? 0 : turn - kSlots + 1); }

  uint32_t *arrived_words(size_t at) const {
    return reinterpret_cast<uint32_t *>(ring + kRingBytes) + at % kRingCount / piece * kTransferBlocks;
  }
  bool has_arrived(size_t p) const {
    const size_t at = p * piece;
    const uint32_t want = value_of(at / kSlotCount);
    const uint32_t *words = arrived_words(at);
    for (unsigned b = 0; b < blocks; ++b)
      if (__atomic_load_n(words + b, __ATOMIC_ACQUIRE) != want) return false;
    return true;
  }
  void move(size_t p) {
    const size_t at = p * piece, n = std::min(piece, count - at);
    unpack(dst + 4 * at, ring + at % kRingCount * width, n, width);
    left[at / kSlotCount].fetch_sub(n, std::memory_order_release);
    done.fetch_add(n, std::memory_order_release);
  }
  // a helper's share: pieces until none is left
  void help() {
    while (true) {
      const size_t p = next_piece.fetch_add(1);
      if (p >= pieces) return;
      Spin spin;
      while (!commit.load(std::memory_order_acquire) || !has_arrived(p)) {
        if (stop.load(std::memory_order_relaxed)) return;
        spin();
      }
      move(p);
    }
  }
};

// The helper threads: up to eight for the process, asleep between copies,
// started by the first copy that wants them and given back with the last
// handle.  They serve every copy that is under way.
struct Helpers {
  std::mutex m;
  std::condition_variable wake, idle;
  std::vector<CopyOut::Job *> jobs;
  std::vector<std::thread> threads;
  bool quit = false;

  void run() {
    std::unique_lock<std::mutex> lock(m);
    while (!quit) {
      CopyOut::Job *hot = nullptr, *cold = nullptr;
      for (CopyOut::Job *j : jobs) {
        if (j->hot && j->next_piece.load() < j->pieces) hot = j;
        if (j->next_fault < j->bytes) cold = j;
      }
      if (hot) {
        ++hot->users;
        lock.unlock();
        hot->help();
        lock.lock();
        if (--hot->users == 0) idle.notify_all();
      } else if (cold) {
        const size_t at = cold->next_fault;
        cold->next_fault += kFaultBytes;
        ++cold->users;
        lock.unlock();
        fault_in(cold->dst + at, std::min(kFaultBytes, cold->bytes - at));
        lock.lock();
        if (--cold->users == 0) idle.notify_all();
      } else {
        wake.wait(lock);
      }
    }
  }
  void add(CopyOut::Job *j) {
    const int cpus = static_cast<int>(std::thread::hardware_concurrency());
    const size_t want = static_cast<size_t>(std::max(1, std::min(kMaxHelpers, cpus / 2)));
    std::lock_guard<std::mutex> lock(m);
    while (threads.size() < want) {
      try {
        threads.emplace_back([this] { run(); });
      } catch (...) {  // fewer helpers then
        break;
      }
    }
    j->listed = true;
    jobs.push_back(j);
    wake.notify_all();
  }
  void heat(CopyOut::Job *j) {
    std::lock_guard<std::mutex> lock(m);
    j->hot = true;
    j->next_fault = j->bytes;  // what is left of the pages the copy takes
    wake.notify_all();
  }
  // returns when no helper touches the job
  void remove(CopyOut::Job *j) {
    std::unique_lock<std::mutex> lock(m);
    if (!j->listed) return;
    jobs.erase(std::find(jobs.begin(), jobs.end(), j));
    idle.wait(lock, [&] { return j->users == 0; });
  }
  void end() {
    std::vector<std::thread> mine;
    {
      std::lock_guard<std::mutex> lock(m);
      quit = true;
      wake.notify_all();
      mine.swap(threads);
    }
    for (std::thread &t : mine) t.join();
    std::lock_guard<std::mutex> lock(m);
    quit = false;
  }
};

namespace {
// (never destroyed: a process may end with handles open and helpers asleep)
Helpers &helpers() {
  static Helpers *h = new Helpers;
  return *h;
}
std::mutex g_handles;  // retain, release and the helpers' end
}  // namespace

CopyOut::CopyOut(uint32_t *dst, size_t count, uint64_t bound) {
  if (!dst || !count) return;
  std::unique_ptr<Job> j(new Job);
  j->dst = reinterpret_cast<char *>(dst);
  j->count = count;
  j->bytes = 4 * count;
  j->width = bound <= 1ull << 16 ? 2 : bound <= 1ull << 24 && count > kHelpersMin ? 3 : 4;
  j->piece = count > kRingCount ? kLargePiece : kPiece;
  j->pieces = (count + j->piece - 1) / j->piece;
  j->blocks = static_cast<unsigned>(std::min<size_t>(kTransferBlocks, (count + 1023) / 1024));
  j->left.reset(new std::atomic<size_t>[j->slot_turns()]);
  for (size_t t = 0; t < j->slot_turns(); ++t) j->left[t] = std::min(kSlotCount, count - t * kSlotCount);
  if (count > kHelpersMin) helpers().add(j.get());
  job_ = j.release();
}

CopyOut::~CopyOut() {
  if (!job_) return;
  job_->stop = true;
  helpers().remove(job_);
  if (queued_) (void)hipStreamSynchronize(stream_);  // no transfer into the ring is left in the stream
  if (job_->ring) ring_return();
  delete job_;
}

// The next transfer: the whole ring at first, then a slot at a time.
void CopyOut::issue() {
  Job &j = *job_;
  const size_t n = std::min(j.issued ? kSlotCount : kRingCount, j.count - j.issued);
  const uint32_t value = j.value_of(j.issued / kSlotCount);
  auto kernel = j.width == 2 ? k_transfer<2> : j.width == 3 ? k_transfer<3> : k_transfer<4>;
  queued_ = true;
  hipLaunchKernelGGL(kernel, dim3(j.blocks), dim3(kBlock), 0, stream_, j.ring + j.issued % kRingCount * j.width,
                     src_ + j.issued, n, j.piece, j.arrived_words(j.issued), value);
  KC_LAUNCH_CHECK();
  g_ring.value = value;
  j.issued += n;
}

void CopyOut::enqueue(const uint32_t *src, hipStream_t stream) {
  if (!job_) return;
  Job &j = *job_;
  if (!j.ring) j.ring = ring_borrow();
  if (!j.ring) return;
  j.first_value = g_ring.value + 1;
  j.issued = 0;  // (also for a call that starts over)
  src_ = src;
  stream_ = stream;
  issue();
  if (!j.listed)
    fault_in(j.dst, j.bytes);
  else if (!j.hot)
    helpers().heat(&j);
}

void CopyOut::finish(const uint32_t *src, hipStream_t stream) {
  if (!job_) return;
  Job &j = *job_;
  if (!queued_) enqueue(src, stream);
  if (!queued_) {  // another copy holds the ring
    KC_HIP(hipMemcpyAsync(j.dst, src, j.bytes, hipMemcpyDeviceToHost, stream));
    KC_HIP(hipStreamSynchronize(stream));
    return;
  }
  j.commit.store(true, std::memory_order_release);
  Spin spin;
  int idle = 0;
  auto looked = std::chrono::steady_clock::now();
  while (j.done.load(std::memory_order_acquire) < j.count) {
    // (only this thread talks to the runtime)
    while (j.issued < j.count && j.left[j.issued / kSlotCount - kSlots].load(std::memory_order_acquire) == 0) issue();
    size_t p = j.next_piece.load();
    if (p < j.pieces && p * j.piece < j.issued && j.has_arrived(p)) {
      if (j.next_piece.compare_exchange_strong(p, p + 1)) j.move(p);
      spin.turns = idle = 0;
      continue;
    }
    spin();
    if (spin.turns % 1024 == 0) {
      const auto now = std::chrono::steady_clock::now();
      if (now - looked > std::chrono::milliseconds(2)) {  // a fault ends the wait
        const hipError_t e = hipStreamQuery(stream);
        if (e != hipErrorNotReady) KC_HIP(e);
        idle = e == hipSuccess ? idle + 1 : 0;
        if (idle > 500) fail(KC_ERR_HIP, "internal: the stream is idle and labels did not arrive");
        looked = now;
      }
    }
  }
  queued_ = false;  // every transfer has arrived
}

void copy_out_retain() {
  std::lock_guard<std::mutex> order(g_handles);
  std::lock_guard<std::mutex> lock(g_ring.m);
  ++g_ring.handles;
}

void copy_out_release() {
  std::lock_guard<std::mutex> order(g_handles);
  {
    std::lock_guard<std::mutex> lock(g_ring.m);
    if (--g_ring.handles > 0) return;
    if (!g_ring.lent) ring_drop();
  }
  helpers().end();
}

}  // namespace kc

// hostcopy.hpp - results from the device into the caller's ordinary memory.  The
// runtime's own copy of pageable memory moves 16 GB/s here: one thread copies out of
// a staging buffer and takes the page faults of a fresh destination (0.2-1 us each).
// HostCopy sends the bytes through a pinned ring in chunks at the link's 56 GB/s, and
// up to kHelpers threads besides the caller take pieces of a chunk: they touch the
// piece's pages while it is on its way and copy it on when it is there.  40 MB into a
// fresh array 3.85 -> 1.23 ms (two helpers 1.26, one 1.66, none 2.92; 512 KB chunks
// 2.0, as a chunk costs the link some 17 us).
//
// Only the caller waits for the stream's earlier work: until the first chunk is there
// a helper sleeps behind its first piece's pages.  (While the helpers waited too, a
// render of 0.63 s that returns 42 MB took 2.53 s of processor time, now 0.64 s.)
//
// The ring (at most kRing bytes) and the helpers belong to the one engine of the
// process, whose calls are serialised: one copy at a time, and a copy is over when
// copy() returns.  The helpers sleep between copies and hold no reference to one that
// is over.
#pragma once
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cerrno>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace nm {

class HostCopy {
 public:
  static constexpr size_t kRing = (size_t)32 << 20;
  // Up to here the runtime's copy.  Whole calls that return 0.5 MB into memory in use:
  // 100 us with it, 106 with the ring; 0.75 MB 112 and 116; 1 MB 137 and 125.  1.2 MB
  // into memory in use or a fresh array: 153 and 403, 135 and 191; 2.8 MB 233 and 711,
  // 178 and 319; 6.2 MB 425 and 930, 295 and 500.
  static constexpr size_t kDirect = (size_t)1 << 20;
  static constexpr int kHelpers = 3;
  // What a thread takes at a time (128 KB of 512 KB chunks: 217 and 549 us); a large
  // result, whose fresh pages come 2 MB at a time, goes by whole chunks (41 MB: 1.80 ->
  // 1.53 ms a call; into memory in use 48 MB 1.70 -> 1.41, 24 MB 0.90 -> 0.80, 16 MB
  // 0.64 -> 0.57, 8 MB 0.37 either way, 4 MB 0.24 -> 0.27: the line could be lower).
  static constexpr size_t kPiece = (size_t)256 << 10;

  // dst[0, bytes) = src (device), after the stream's earlier work; returns when the
  // bytes are there (or with the first error, when no thread touches dst any more)
  hipError_t copy(hipStream_t stream, void* dst, const void* src, size_t bytes) {
    if (bytes <= kDirect || registered(dst) || !prepare(bytes)) {
      const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
      return e == hipSuccess ? hipStreamSynchronize(stream) : e;
    }
    const bool large = bytes >= ((size_t)24 << 20);
    const size_t chunk = large ? (size_t)2 << 20 : (size_t)1 << 20, piece = large ? chunk : kPiece;
    const int n = (int)((bytes + chunk - 1) / chunk), slots = (int)std::min<size_t>(ring_ / chunk, kEvents);
    const int per = (int)(chunk / piece);
    Job j;
    j.dst = (char*)dst;
    j.ring = (const char*)pinned_;
    j.bytes = bytes;
    j.piece = piece;
    j.per = per;
    j.slots = slots;
    j.events = events_.data();
    std::vector<std::atomic<int>> done((size_t)n);  // pieces of each chunk that left the ring
    j.done = done.data();
    open(&j, kHelpers);
    hipError_t err = hipSuccess;
    for (int i = 0; i < n && err == hipSuccess; i++) {
      // the slot's previous chunk must have left it; meanwhile this thread helps
      if (i >= slots) arrive(j);
      while (i >= slots && j.done[i - slots].load(std::memory_order_acquire) < per)
        if (!step(j, true)) std::this_thread::yield();
      if (j.error.load() != hipSuccess) break;
      const size_t o = (size_t)i * chunk;
      err = hipMemcpyAsync((char*)pinned_ + (size_t)(i % slots) * chunk, (const char*)src + o, std::min(chunk, bytes - o),
                           hipMemcpyDeviceToHost, stream);
      if (err == hipSuccess) err = hipEventRecord(events_[i % slots], stream);
      if (err == hipSuccess)
        j.issued.store((int)std::min<size_t>((size_t)(i + 1) * per, (bytes + piece - 1) / piece),
                       std::memory_order_release);
    }
    if (err != hipSuccess) j.error.store(err);
    j.closed.store(true, std::memory_order_release);
    while (step(j, true)) {
    }
    arrive(j);  // the helpers took every piece
    close(&j);  // every helper has left the job
    err = (hipError_t)j.error.load();
    const hipError_t s = hipStreamSynchronize(stream);
    return err != hipSuccess ? err : s;
  }

 private:
  static constexpr int kEvents = 64;

  struct Job {
    char* dst = nullptr;
    const char* ring = nullptr;
    size_t bytes = 0, piece = 0;
    int per = 0, slots = 0;  // pieces of a chunk, chunks of the ring
    const hipEvent_t* events = nullptr;
    std::atomic<int>* done = nullptr;
    std::atomic<int> next{0}, issued{0}, error{hipSuccess};
    std::atomic<bool> closed{false};
    std::atomic<bool> arrived{false};  // the first chunk is there (or never will be)
    int inside = 0;  // helpers in the job (HostCopy::mu_)

    bool over() const { return closed.load(std::memory_order_acquire) && next.load() >= issued.load(); }
  };

  // copies one piece on; false: none is issued that nobody has taken
  bool step(Job& j, bool caller) {
    int i = j.next.load(std::memory_order_relaxed);
    do {
      if (i >= j.issued.load(std::memory_order_acquire)) return false;
    } while (!j.next.compare_exchange_weak(i, i + 1));
    const int c = i / j.per, slot = c % j.slots;
    const size_t o = (size_t)i * j.piece, size = std::min(j.piece, j.bytes - o);
    hipError_t e = j.error.load() == hipSuccess ? hipSuccess : hipErrorUnknown;
    if (e == hipSuccess) {
      populate(j.dst + o, size);
      if (caller) {
        arrive(j);
      } else if (!j.arrived.load(std::memory_order_acquire)) {
        std::unique_lock<std::mutex> lk(mu_);
        first_.wait(lk, [&] { return j.arrived.load(); });
      }
      e = hipEventSynchronize(j.events[slot]);
    }
    if (e == hipSuccess) std::memcpy(j.dst + o, j.ring + ((size_t)slot * j.per + i % j.per) * j.piece, size);
    else if (j.error.load() == hipSuccess) j.error.store(e);
    j.done[c].fetch_add(1, std::memory_order_release);
    return true;
  }
  // the caller waits for the first chunk (if it was sent), then wakes the helpers
  void arrive(Job& j) {
    if (j.arrived.load()) return;
    if (j.issued.load() > 0) {
      const hipError_t e = hipEventSynchronize(j.events[0]);
      if (e != hipSuccess && j.error.load() == hipSuccess) j.error.store(e);
    }
    std::lock_guard<std::mutex> lk(mu_);
    j.arrived.store(true, std::memory_order_release);
    first_.notify_all();
  }

  // the pages of a destination that nobody has touched yet, while its bytes are on
  // their way; without the call (Linux before 5.14) the copy takes the faults
  static void populate(char* p, size_t n) {
#ifdef MADV_POPULATE_WRITE
    constexpr uintptr_t page = 4096;
    const uintptr_t a = ((uintptr_t)p + page - 1) & ~(page - 1), b = ((uintptr_t)p + n) & ~(page - 1);
    if (b > a) {
      const int keep = errno;
      (void)madvise((void*)a, b - a, MADV_POPULATE_WRITE);
      errno = keep;
    }
#else
    (void)p;
    (void)n;
#endif
  }

  // memory the runtime knows (pinned, managed, a device's): its own copy goes there at
  // the link's rate by itself (66 MB into pinned memory 1.37 ms a call, by the ring
  // 1.88), and a device's is nothing for a thread to write to
  static bool registered(const void* dst) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, dst) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
  }

  // the ring and its events, and the helpers (once); false: do without
  bool prepare(size_t bytes) {
    const size_t want = std::min(kRing, (bytes + ((size_t)4 << 20)) & ~(((size_t)2 << 20) - 1));
    if (want > ring_) {
      if (pinned_) (void)hipHostFree(pinned_);
      pinned_ = nullptr;
      ring_ = 0;
      if (hipHostMalloc(&pinned_, want, hipHostMallocDefault) != hipSuccess) {
        pinned_ = nullptr;
        (void)hipGetLastError();
        return false;
      }
      ring_ = want;
    }
    while ((int)events_.size() < kEvents) {
      hipEvent_t e = nullptr;
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      events_.push_back(e);
    }
    if (!started_) {
      started_ = true;
      const int spare = (int)std::thread::hardware_concurrency() - 1;
      try {
        for (int t = 0; t < std::min(kHelpers, spare); t++) std::thread([this] { help(); }).detach();
      } catch (...) {  // no thread to be had: the caller copies alone
      }
    }
    return true;
  }

  void open(Job* j, int helpers) {
    std::lock_guard<std::mutex> lk(mu_);
    job_ = j;
    wanted_ = helpers;
    if (helpers > 0) cv_.notify_all();
  }
  void close(Job* j) {
    std::unique_lock<std::mutex> lk(mu_);
    job_ = nullptr;
    left_.wait(lk, [&] { return j->inside == 0; });
  }
  void help() {
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      cv_.wait(lk, [&] { return job_ != nullptr && wanted_ > 0; });
      Job* j = job_;
      wanted_--;
      j->inside++;
      lk.unlock();
      while (!j->over())
        if (!step(*j, false)) std::this_thread::yield();
      lk.lock();
      if (--j->inside == 0) left_.notify_all();
    }
  }

  void* pinned_ = nullptr;
  size_t ring_ = 0;
  std::vector<hipEvent_t> events_;
  bool started_ = false;
  std::mutex mu_;
  std::condition_variable cv_, left_, first_;
  Job* job_ = nullptr;
  int wanted_ = 0;
};

}  // namespace nm

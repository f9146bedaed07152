// transfer.hpp -- large copies between a caller's pageable host memory and the
// GPU.
//
// The runtime's own copy of pageable memory stages it through its pinned
// buffers with one host thread: about 6 GB/s for a field read into fresh
// memory, whose pages that thread also faults in (134 MB, a 4096^2 field:
// 22 ms, as long as 20 of its time steps).  Here the copy engine moves
// chunks between the device and a pinned ring while a few host threads, each
// a chunk at a time, move them between the ring and the caller's memory.
//
// One ring and one pool of threads per process, made at the first large
// copy: 32 MiB pinned and at most 7 threads, asleep between copies.  A copy
// that finds them in use by another thread, or whose host pointer the runtime
// already knows (pinned, managed or device memory), takes the runtime's path.
// So does a download of less than 8 MiB or an upload of less than 48 MiB, where
// waking the threads and a call per chunk cost more than they save: the
// runtime copies from the device into memory at 8 to 19 GB/s but reads resident
// memory at 30.  Both paths measured, us by the runtime and here: downloads
// of 4.5 MiB 270 / 288, 6 MiB 364 / 364, 8 MiB 482 / 407, 32 MiB 1950 / 963 (into
// fresh memory 3460 / 1230), 128 MiB 7770 / 3470; uploads of 4.5 MiB 176 / 294,
// 8 MiB 268 / 427, 32 MiB 1006 / 1034, 48 MiB 1735 / 1493, 64 MiB 2420 / 1911, 128 MiB 4706 / 3599.
//
// The threads are joined when the process ends normally or the library is
// unloaded; later copies (by destructors that run after that) take the
// runtime's path, as do those of a forked child, which has the ring but none
// of the threads.  The object itself is never destroyed: a condition variable
// that threads of the parent wait on must not be destroyed in the child (the
// destructor waits for them), and late callers may still use the rest.
#pragma once
#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace fsibe {

class Transfer {
 public:
  static Transfer &get() {
    static Transfer *t = new Transfer;
    static struct End {
      ~End() { t->stop(); }
    } end;
    return *t;
  }
  // download returns when the data are in place; upload when the source may be
  // reused, or, where the runtime's path is taken, as hipMemcpyAsync does
  hipError_t download(void *dst, const void *src, size_t bytes, hipStream_t st) { return copy(dst, src, bytes, st, false); }
  hipError_t upload(void *dst, const void *src, size_t bytes, hipStream_t st) { return copy(dst, src, bytes, st, true); }

 private:
  Transfer() = default;

  // ends the helpers; the pinned ring stays until the process ends (the
  // runtime may be gone)
  void stop() {
    if (pid_ != getpid()) return;  // a forked child: the threads are not there
    // held by a copy of another thread that the process's end cuts short: its
    // helpers end with the process
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (!use.owns_lock()) return;
    {
      std::lock_guard<std::mutex> g(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto &w : workers_) w.join();
    workers_.clear();
  }

  static constexpr size_t kMinDown = (size_t)8 << 20, kMinUp = (size_t)48 << 20;
  static constexpr size_t kSlot = 2 << 20;  // largest chunk: a huge page, faulted in by one thread
  static constexpr int kSlots = 16, kHelpers = 7;

  hipError_t plain(void *dst, const void *src, size_t bytes, hipStream_t st, bool up) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st);
    return e != hipSuccess || up ? e : hipStreamSynchronize(st);
  }

  // the ring and the helpers, made at the first use (also while some other
  // thread captures a graph); the caller holds use_
  bool ready() {
    if (stop_) return false;
    if (ring_) return pid_ == getpid();
    if (failed_) return false;
    failed_ = true;
    void *p = nullptr;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool sw = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    const hipError_t e = hipHostMalloc(&p, kSlots * kSlot, hipHostMallocPortable);
    if (sw) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    const int hw = (int)std::thread::hardware_concurrency();
    const int n = std::min(kHelpers, std::max(0, hw / 2 - 1));
    try {
      for (int i = 0; i < n; ++i) workers_.emplace_back([this] { loop(); });
    } catch (...) {  // fewer helpers than wanted: the ones that started serve
    }
    ring_ = (char *)p;
    pid_ = getpid();
    failed_ = false;
    return true;
  }

  hipError_t copy(void *dst, const void *src, size_t bytes, hipStream_t st, bool up) {
    if (bytes < (up ? kMinUp : kMinDown)) return plain(dst, src, bytes, st, up);
    hipPointerAttribute_t at;
    const hipError_t known = hipPointerGetAttributes(&at, up ? src : dst);
    if (known != hipSuccess) (void)hipGetLastError();
    if (known == hipSuccess && at.type != hipMemoryTypeUnregistered) return plain(dst, src, bytes, st, up);
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (!use.owns_lock() || !ready()) return plain(dst, src, bytes, st, up);
    Job j;
    j.host = up ? (char *)const_cast<void *>(src) : (char *)dst;
    j.dev = up ? (char *)dst : (char *)const_cast<void *>(src);
    j.bytes = bytes;
    j.chunk = std::min(kSlot, std::max(bytes / 12 >> 16 << 16, (size_t)512 << 10));
    // the first chunk ends where the others are aligned
    j.lead = j.chunk - (size_t)((uintptr_t)j.host % j.chunk);
    j.n = 1 + (long)((bytes - std::min(bytes, j.lead) + j.chunk - 1) / j.chunk);
    j.up = up;
    const int slots = (int)std::min<long>(j.n, kSlots);
    hipEvent_t ev[kSlots];
    int nev = 0;
    hipError_t e = hipSuccess;
    while (nev < slots && e == hipSuccess)
      if ((e = hipEventCreateWithFlags(&ev[nev], hipEventDisableTiming)) == hipSuccess) ++nev;
    if (e == hipSuccess) {
      start(j);
      // chunk i uses slot i % kSlots once chunk i - kSlots has left it
      long issued = 0, ready = 0;  // device copies issued; chunks the helpers may move
      auto moved = [&](long i) { return slot_done_[i % kSlots].load(std::memory_order_acquire) >= i + 1; };
      auto landed = [&](long i) {  // chunk i's device copy is over (or has failed: e)
        const hipError_t q = hipEventQuery(ev[i % kSlots]);
        if (q != hipSuccess && q != hipErrorNotReady) e = q;
        return q == hipSuccess;
      };
      auto issue = [&](long i) {
        char *r = ring_ + (size_t)(i % kSlots) * kSlot, *d = j.dev + j.begin(i);
        e = up ? hipMemcpyAsync(d, r, j.len(i), hipMemcpyHostToDevice, st)
               : hipMemcpyAsync(r, d, j.len(i), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev[i % kSlots], st);
      };
      while (e == hipSuccess && (up ? issued : ready) < j.n) {
        bool any = false;
        if (up) {
          if (ready < j.n && (ready < kSlots || (ready - kSlots < issued && landed(ready - kSlots)))) ++ready, any = true;
          if (issued < ready && moved(issued)) issue(issued++), any = true;
        } else {
          if (issued < j.n && (issued < kSlots || moved(issued - kSlots))) issue(issued++), any = true;
          if (e == hipSuccess && ready < issued && landed(ready)) ++ready, any = true;
        }
        if (any) published_.store(ready, std::memory_order_release);
        else if (!workers_.empty() || !help()) std::this_thread::yield();
      }
      if (e == hipSuccess && !up)
        for (long i = std::max(0L, j.n - kSlots); i < j.n; ++i)
          while (!moved(i))
            if (!help()) std::this_thread::yield();
      end();
      // no device copy from or into the ring outlives the call
      const hipError_t q = hipStreamSynchronize(st);
      if (e == hipSuccess) e = q;
    }
    for (int i = 0; i < nev; ++i) (void)hipEventDestroy(ev[i]);
    if (e == hipSuccess) (void)hipGetLastError();  // an event query's "not ready" is no error of the caller's
    return e;
  }

  // ---- host copies: a chunk at a time, taken by whoever is free
  struct Job {
    char *host, *dev;
    size_t bytes, chunk, lead;
    long n;
    bool up;
    size_t begin(long i) const { return i == 0 ? 0 : std::min(bytes, lead + (size_t)(i - 1) * chunk); }
    size_t len(long i) const { return begin(i + 1) - begin(i); }
  };
  void start(const Job &j) {
    job_ = j;
    published_.store(0);
    next_.store(0);
    over_.store(false);
    for (auto &d : slot_done_) d.store(0);
    {
      std::lock_guard<std::mutex> g(mu_);
      active_ = (int)workers_.size();
      ++gen_;
    }
    cv_.notify_all();
  }
  // moves the next published chunk; false if there is none
  bool help() {
    long i = next_.load();
    do {
      if (i >= published_.load(std::memory_order_acquire)) return false;
    } while (!next_.compare_exchange_weak(i, i + 1));
    char *h = job_.host + job_.begin(i), *r = ring_ + (size_t)(i % kSlots) * kSlot;
    if (job_.up) memcpy(r, h, job_.len(i));
    else memcpy(h, r, job_.len(i));
    slot_done_[i % kSlots].store(i + 1, std::memory_order_release);
    return true;
  }
  void end() {
    over_.store(true, std::memory_order_release);
    std::unique_lock<std::mutex> g(mu_);
    done_.wait(g, [this] { return active_ == 0; });
  }
  void loop() {
    unsigned long long seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> g(mu_);
        cv_.wait(g, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
      }
      // until all chunks are taken, or the copy failed
      while (!over_.load(std::memory_order_acquire) && next_.load() < job_.n)
        if (!help()) std::this_thread::yield();
      std::lock_guard<std::mutex> g(mu_);
      if (--active_ == 0) done_.notify_one();
    }
  }

  std::mutex use_, mu_;
  std::condition_variable cv_, done_;
  std::vector<std::thread> workers_;
  char *ring_ = nullptr;
  bool failed_ = false, stop_ = false;
  pid_t pid_ = getpid();
  unsigned long long gen_ = 0;
  int active_ = 0;
  Job job_{};
  std::atomic<long> published_{0}, next_{0};
  std::atomic<long> slot_done_[kSlots] = {};  // 1 + the last chunk moved through the slot
  std::atomic<bool> over_{false};
};

}  // namespace fsibe

// transfer.hpp -- copies between a caller's pageable host memory and the GPU.
//
// The runtime's own copy of pageable memory stages it through its pinned
// buffers with one host thread: about 6 GB/s for a field read into fresh
// memory, whose pages that thread also faults in (134 MB, a 4096^2 field:
// 22 ms, as long as 20 of its time steps).  Here the copy engine moves
// chunks between the device and a pinned ring while a few host threads move
// them between the ring and the caller's memory.
//
// One ring and one pool of threads per process, made at the first large
// copy: at most 16 MiB pinned and 7 threads, asleep between copies.  A copy
// that finds them in use by another thread, or whose host pointer the runtime
// already knows (pinned, managed or device memory), takes the runtime's path,
// as does a small one.
#pragma once
#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace fsibe {

class Transfer {
 public:
  static Transfer &get() {
    static Transfer t;
    return t;
  }
  // download returns when the data are in place; upload when the source may be
  // reused, or, where the runtime's path is taken, as hipMemcpyAsync does
  hipError_t download(void *dst, const void *src, size_t bytes, hipStream_t st) { return copy(dst, src, bytes, st, false); }
  hipError_t upload(void *dst, const void *src, size_t bytes, hipStream_t st) { return copy(dst, src, bytes, st, true); }

  ~Transfer() {
    if (pid_ != getpid()) {  // a forked child: the threads are not there
      new std::vector<std::thread>(std::move(workers_));
      return;
    }
    {
      std::lock_guard<std::mutex> g(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto &w : workers_) w.join();
    // the pinned ring stays until the process ends: the runtime may be gone
  }

 private:
  static constexpr size_t kMin = 192 << 10;   // below, the runtime's path is as fast
  static constexpr size_t kUnit = 64 << 10;   // one host copy
  static constexpr size_t kSlot = 2 << 20;    // largest chunk (one device copy)
  static constexpr int kSlots = 8, kHelpers = 7;

  hipError_t plain(void *dst, const void *src, size_t bytes, hipStream_t st, bool up) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st);
    return e != hipSuccess || up ? e : hipStreamSynchronize(st);
  }

  // the ring and the helpers, made at the first use (also while some other
  // thread captures a graph)
  bool ready() {
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
    if (bytes < kMin) return plain(dst, src, bytes, st, up);
    hipPointerAttribute_t at;
    const hipError_t known = hipPointerGetAttributes(&at, up ? src : dst);
    if (known != hipSuccess) (void)hipGetLastError();
    if (known == hipSuccess && at.type != hipMemoryTypeUnregistered) return plain(dst, src, bytes, st, up);
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (!use.owns_lock() || !ready()) return plain(dst, src, bytes, st, up);
    // about six chunks of a small copy, so that both halves of the way are busy
    const size_t chunk = std::min(kSlot, std::max((bytes / 6 + kUnit - 1) / kUnit, (size_t)2) * kUnit);
    const long n = (long)((bytes + chunk - 1) / chunk);
    const int slots = (int)std::min<long>(n, kSlots);
    hipEvent_t ev[kSlots];
    int nev = 0;
    hipError_t e = hipSuccess;
    while (nev < slots && e == hipSuccess)
      if ((e = hipEventCreateWithFlags(&ev[nev], hipEventDisableTiming)) == hipSuccess) ++nev;
    if (e == hipSuccess) {
      auto len = [&](long i) { return std::min(chunk, bytes - (size_t)i * chunk); };
      auto slot = [&](long i) { return ring_ + (size_t)(i % kSlots) * kSlot; };
      start(Job{up ? (char *)const_cast<void *>(src) : (char *)dst, bytes, chunk, up});
      if (up) {
        for (long i = 0; i < n && e == hipSuccess; ++i) {
          if (i >= kSlots) e = hipEventSynchronize(ev[i % kSlots]);  // the slot's last chunk is on the device
          if (e != hipSuccess) break;
          move_chunk(i);
          e = hipMemcpyAsync((char *)dst + (size_t)i * chunk, slot(i), len(i), hipMemcpyHostToDevice, st);
          if (e == hipSuccess) e = hipEventRecord(ev[i % kSlots], st);
        }
      } else {
        long issued = 0;
        for (long i = 0; i < n && e == hipSuccess; ++i) {
          // chunk issued - kSlots has left its slot: move_chunk returned for it
          for (; issued < n && issued < i + kSlots && e == hipSuccess; ++issued) {
            e = hipMemcpyAsync(slot(issued), (const char *)src + (size_t)issued * chunk, len(issued),
                               hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ev[issued % kSlots], st);
          }
          if (e == hipSuccess) e = hipEventSynchronize(ev[i % kSlots]);
          if (e == hipSuccess) move_chunk(i);
        }
      }
      end();
      // no device copy from or into the ring outlives the call
      const hipError_t s = hipStreamSynchronize(st);
      if (e == hipSuccess) e = s;
    }
    for (int i = 0; i < nev; ++i) (void)hipEventDestroy(ev[i]);
    return e;
  }

  // ---- host copies: units of a chunk, taken by whoever is free
  struct Job {
    char *host;
    size_t bytes, chunk;
    bool up;
    long units() const { return (long)((bytes + kUnit - 1) / kUnit); }
    long per_chunk() const { return (long)(chunk / kUnit); }
  };
  void start(const Job &j) {
    job_ = j;
    published_.store(0);
    next_.store(0);
    moved_.store(0);
    over_.store(false);
    {
      std::lock_guard<std::mutex> g(mu_);
      active_ = (int)workers_.size();
      ++gen_;
    }
    cv_.notify_all();
  }
  void move_unit(long u) {
    const size_t off = (size_t)u * kUnit, len = std::min(kUnit, job_.bytes - off);
    const long i = u / job_.per_chunk();
    char *h = job_.host + off, *r = ring_ + (size_t)(i % kSlots) * kSlot + (off - (size_t)i * job_.chunk);
    if (job_.up) memcpy(r, h, len);
    else memcpy(h, r, len);
    moved_.fetch_add(1, std::memory_order_acq_rel);
  }
  // lets the helpers at chunk i (its slot is ready), takes part, and returns
  // when all units of chunks 0 .. i have been moved (no later unit can have been)
  void move_chunk(long i) {
    const long want = std::min((i + 1) * job_.per_chunk(), job_.units());
    published_.store(want, std::memory_order_release);
    long u = next_.load();
    while (u < want)
      if (next_.compare_exchange_weak(u, u + 1)) {
        move_unit(u);
        u = next_.load();
      }
    while (moved_.load(std::memory_order_acquire) < want) std::this_thread::yield();
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
      const long n = job_.units();
      for (;;) {
        if (over_.load(std::memory_order_acquire)) break;  // nothing left, or the copy failed
        long u = next_.load();
        if (u >= n) break;
        if (u < published_.load(std::memory_order_acquire)) {
          if (next_.compare_exchange_weak(u, u + 1)) move_unit(u);
        } else {
          std::this_thread::yield();
        }
      }
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
  std::atomic<long> published_{0}, next_{0}, moved_{0};
  std::atomic<bool> over_{false};
};

}  // namespace fsibe

// lbm_readback.hpp — device results to caller memory.  Not part of the public ABI.
//
// What bounds a copy into ordinary (pageable) memory is the host: the runtime
// moves it through its own staging on one thread, which also takes the fresh
// pages' faults (10 GB/s measured, 207 ms for the four moment fields of 512^3
// cells).  Here the device writes 2 MiB pinned slots at the link's rate and a
// few threads copy them out, so the faults and the copies run in parallel.
// Results are produced piece by piece through a bounded device workspace, so
// no call allocates a full-size array either.
//
// One object per context; calls on a context are serialized by the caller,
// different contexts share nothing.  The pinned slots and the workspace are
// allocated at first use, bounded (kSlots * kSlotBytes, kWorkBytes) and given
// back with the context.  Threads live only inside a call.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

class Readback {
 public:
  struct Seg {
    void* dst;
    const void* src;
    size_t bytes;
  };
  static constexpr size_t kSlotBytes = (size_t)2 << 20;
  static constexpr int kSlots = 24;
  static constexpr size_t kWorkBytes = (size_t)64 << 20;
  static constexpr int kThreads = 12;  // of the 16 host cores a GPU comes with

  Readback() = default;
  Readback(const Readback&) = delete;
  Readback& operator=(const Readback&) = delete;
  ~Readback() {
    for (hipEvent_t e : ev_) (void)hipEventDestroy(e);
    if (pin_) (void)hipHostFree(pin_);
    if (work_) (void)hipFree(work_);
  }

  // Device workspace of kWorkBytes for the pieces; null when it cannot be had.
  void* work() {
    if (!work_ && hipMalloc(&work_, kWorkBytes) != hipSuccess) work_ = nullptr;
    return work_;
  }

  // Runs produce(p, segs) for p = 0 .. pieces - 1 in order.  Each call enqueues
  // what fills its sources on `s` and lists the segments to copy; on return
  // every destination is filled.  Pieces may reuse one source buffer: copies
  // and producers are in the stream's order.
  hipError_t read(int device, hipStream_t s, int pieces,
                  const std::function<hipError_t(int, std::vector<Seg>&)>& produce) {
    std::vector<Seg> segs;
    segs.reserve(64);  // nothing is allocated while threads run
    hipError_t e = hipSuccess;
    if (!ensure_slots()) {  // no pinned memory: the runtime's own copies
      for (int p = 0; p < pieces && e == hipSuccess; ++p) {
        segs.clear();
        e = produce(p, segs);
        for (const Seg& g : segs)
          if (e == hipSuccess) e = hipMemcpyAsync(g.dst, g.src, g.bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
      }
      return e;
    }
    Job job;
    std::vector<std::thread> pool;
    pool.reserve(kThreads);
    for (int p = 0; p < pieces && e == hipSuccess; ++p) {
      segs.clear();
      e = produce(p, segs);
      if (e != hipSuccess) break;
      size_t total = 0;
      for (const Seg& g : segs) total += g.bytes;
      if (pieces == 1 && total <= kSlotBytes) {  // one slot, one wait, no thread
        size_t at = 0;
        for (const Seg& g : segs) {
          if (e == hipSuccess) e = hipMemcpyAsync(pin_ + at, g.src, g.bytes, hipMemcpyDeviceToHost, s);
          at += g.bytes;
        }
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        at = 0;
        for (const Seg& g : segs) {
          if (e == hipSuccess) memcpy(g.dst, pin_ + at, g.bytes);
          at += g.bytes;
        }
        return e;
      }
      if (pool.empty()) {
        // A thread that cannot be had is done without: the caller's own
        // thread drains the queue when no worker exists.
        const int want = (int)std::min<size_t>(kThreads, (pieces * total + kSlotBytes - 1) / kSlotBytes);
        try {
          for (int t = 0; t < want; ++t) pool.emplace_back([this, device, &job] { worker(device, job); });
        } catch (...) {
        }
      }
      for (const Seg& g : segs)
        for (size_t at = 0; at < g.bytes && e == hipSuccess; at += kSlotBytes) {
          const size_t n = std::min(kSlotBytes, g.bytes - at);
          const int k = job.take(pool.empty() ? this : nullptr);
          e = hipMemcpyAsync(pin_ + (size_t)k * kSlotBytes, (const char*)g.src + at, n, hipMemcpyDeviceToHost, s);
          if (e == hipSuccess) e = hipEventRecord(ev_[k], s);
          if (e == hipSuccess) job.put(Item{k, (char*)g.dst + at, n});
        }
    }
    job.close();
    if (pool.empty()) worker(device, job);
    for (std::thread& t : pool) t.join();
    // nothing of this call is left on the stream, also after an error
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e != hipSuccess ? e : (hipError_t)job.err.load();
  }

 private:
  struct Item {
    int slot;
    char* dst;
    size_t bytes;
  };
  // free slots and filled ones, each at most kSlots: fixed arrays, so that no
  // thread allocates
  struct Job {
    std::mutex mu;
    std::condition_variable cv;
    int free[kSlots], nfree = kSlots;
    Item queue[kSlots];
    int head = 0, count = 0;
    bool done = false;
    std::atomic<int> err{(int)hipSuccess};
    Job() {
      for (int k = 0; k < kSlots; ++k) free[k] = kSlots - 1 - k;
    }
    Item pop() {
      const Item it = queue[head];
      head = (head + 1) % kSlots;
      --count;
      return it;
    }
    // a free slot; `self`: no worker exists, so drain an item here
    int take(Readback* self) {
      std::unique_lock<std::mutex> lk(mu);
      while (nfree == 0) {
        if (self) {
          const Item it = pop();
          lk.unlock();
          self->drain(it, *this);
          lk.lock();
        } else {
          cv.wait(lk);
        }
      }
      return free[--nfree];
    }
    void put(const Item& it) {
      {
        std::lock_guard<std::mutex> lk(mu);
        queue[(head + count++) % kSlots] = it;
      }
      cv.notify_all();
    }
    void close() {
      {
        std::lock_guard<std::mutex> lk(mu);
        done = true;
      }
      cv.notify_all();
    }
  };

  void drain(const Item& it, Job& job) {
    const hipError_t e = hipEventSynchronize(ev_[it.slot]);
    if (e == hipSuccess)
      memcpy(it.dst, pin_ + (size_t)it.slot * kSlotBytes, it.bytes);
    else
      job.err.store((int)e);
    {
      std::lock_guard<std::mutex> lk(job.mu);
      job.free[job.nfree++] = it.slot;
    }
    job.cv.notify_all();
  }

  void worker(int device, Job& job) {
    (void)hipSetDevice(device);
    for (;;) {
      Item it;
      {
        std::unique_lock<std::mutex> lk(job.mu);
        job.cv.wait(lk, [&] { return job.done || job.count > 0; });
        if (job.count == 0) return;
        it = job.pop();
      }
      drain(it, job);
    }
  }

  bool ensure_slots() {
    if (pin_) return true;
    if (failed_) return false;
    void* p = nullptr;
    if (hipHostMalloc(&p, kSlotBytes * kSlots, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      failed_ = true;
      return false;
    }
    for (int k = 0; k < kSlots; ++k) {
      hipEvent_t e;
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        for (hipEvent_t x : ev_) (void)hipEventDestroy(x);
        ev_.clear();
        (void)hipHostFree(p);
        failed_ = true;
        return false;
      }
      ev_.push_back(e);
    }
    pin_ = (char*)p;
    return true;
  }

  char* pin_ = nullptr;
  std::vector<hipEvent_t> ev_;
  void* work_ = nullptr;
  bool failed_ = false;
};

}  // namespace lbm

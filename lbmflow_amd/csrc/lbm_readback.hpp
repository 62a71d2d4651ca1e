// lbm_readback.hpp — device results to caller memory.  Not part of the public ABI.
//
// What bounds a copy into ordinary (pageable) memory is the host: the runtime
// moves it through its own staging on one thread, which also takes the fresh
// pages' faults (10 GB/s measured, 207 ms for the four moment fields of 512^3
// cells).  Here the device writes 2 MiB pinned slots at the link's rate and a
// few threads copy them out, so the faults and the copies run in parallel.  A
// kernel writes the slots: the runtime's copies go to a DMA engine of its
// choice, and now and then, for a while, to one that takes 166 us per slot
// instead of 42 (32 MB 1.0 or 3.0 ms).
// Results are produced piece by piece through a bounded device workspace, so
// no call allocates a full-size array either.
//
// One object per context; calls on a context are serialized by the caller,
// different contexts share nothing.  The pinned slots and the workspace are
// allocated at first use, as large as the largest read so far needs and at most
// kSlots * kSlotBytes and kWorkBytes, and given back with the context.  Threads
// live only inside a call.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

// n bytes (a multiple of 4, 4-byte aligned) into pinned memory (lbm_kernels.hip)
hipError_t launch_to_host(void* dst, const void* src, size_t n, hipStream_t s);

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
  static constexpr size_t kMinWorkBytes = (size_t)64 << 10;
  // a small array that no kernel has just written is 3 us faster by the runtime's
  // copy (110 KB 12.1 against 15.4 us)
  static constexpr size_t kSmallCopy = (size_t)512 << 10;
  static constexpr int kThreads = 12;  // of the 16 host cores a GPU comes with

  Readback() = default;
  Readback(const Readback&) = delete;
  Readback& operator=(const Readback&) = delete;
  ~Readback() {
    for (hipEvent_t e : ev_) (void)hipEventDestroy(e);
    if (pin_) (void)hipHostFree(pin_);
    if (work_) (void)hipFree(work_);
  }

  // Gives the device workspace back (no read is running); whether there was one.
  bool release_work() {
    const bool had = work_ != nullptr;
    if (had) (void)hipFree(work_);
    work_ = nullptr;
    work_bytes_ = 0;
    return had;
  }

  // `planes` planes of n floats to out(plane).  produce(i0, cnt, w) enqueues on
  // `s` what writes the values i0 .. i0 + cnt - 1 of each plane to w + plane *
  // cnt.  hipErrorOutOfMemory: no workspace could be had.
  hipError_t read_planes(int device, hipStream_t s, uint32_t n, uint32_t planes,
                         const std::function<float*(uint32_t)>& out,
                         const std::function<hipError_t(uint32_t, uint32_t, float*)>& produce) {
    size_t have = 0;
    float* w = (float*)work((size_t)planes * n * sizeof(float), &have);
    if (!w) return hipErrorOutOfMemory;
    size_t per = have / sizeof(float) / planes;
    per = per < n ? per / 64 * 64 : n;
    const int pieces = (int)((n + per - 1) / per);
    return read(device, s, pieces, [&](int p, std::vector<Seg>& segs) {
      const uint32_t i0 = (uint32_t)(p * per), cnt = (uint32_t)std::min<size_t>(per, n - i0);
      for (uint32_t k = 0; k < planes; ++k)
        segs.push_back({out(k) + i0, w + (size_t)k * cnt, (size_t)cnt * sizeof(float)});
      return produce(i0, cnt, w);
    });
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
    bool slots = false;
    Job job;
    std::vector<std::thread> pool;
    pool.reserve(kThreads);
    for (int p = 0; p < pieces && e == hipSuccess; ++p) {
      segs.clear();
      e = produce(p, segs);
      if (e != hipSuccess) break;
      size_t total = 0;
      for (const Seg& g : segs) total += g.bytes;
      const bool one = pieces == 1 && total <= kSlotBytes;
      if (p == 0) slots = ensure_slots(one ? 1 : kSlots);
      if (!slots) {  // no pinned memory: the runtime's own copies
        for (const Seg& g : segs)
          if (e == hipSuccess) e = hipMemcpyAsync(g.dst, g.src, g.bytes, hipMemcpyDeviceToHost, s);
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        continue;
      }
      if (one) {  // one slot, one wait, no thread
        size_t at = 0;
        for (size_t a = 0, b; a < segs.size() && e == hipSuccess; a = b) {
          size_t n = 0;
          for (b = a; b < segs.size() && segs[b].src == (const char*)segs[a].src + n; ++b) n += segs[b].bytes;
          e = segs.size() == 1 && n <= kSmallCopy ? hipMemcpyAsync(pin_ + at, segs[a].src, n, hipMemcpyDeviceToHost, s)
                                                  : launch_to_host(pin_ + at, segs[a].src, n, s);
          at += n;
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
      // one copy per slot, over as many segments as lie together in the
      // source (a DMA copy for each of 19 planes of 24^3 cells took 1.03 ms, one
      // for all 0.07)
      Item it;
      const char* src = nullptr;
      size_t fill = 0;
      auto flush = [&] {
        if (fill == 0 || e != hipSuccess) return;
        it.slot = job.take(pool.empty() ? this : nullptr);
        e = launch_to_host(pin_ + (size_t)it.slot * kSlotBytes, src, fill, s);
        if (e == hipSuccess) e = hipEventRecord(ev_[it.slot], s);
        if (e == hipSuccess) job.put(it);
        fill = 0;
        it.parts = 0;
      };
      for (const Seg& g : segs)
        for (size_t at = 0, n; at < g.bytes && e == hipSuccess; at += n) {
          const char* from = (const char*)g.src + at;
          if (fill && (fill == kSlotBytes || it.parts == kParts || from != src + fill)) flush();
          if (fill == 0) src = from;
          n = std::min(kSlotBytes - fill, g.bytes - at);
          it.part[it.parts++] = {(char*)g.dst + at, n};
          fill += n;
        }
      flush();
    }
    job.close();
    if (pool.empty()) worker(device, job);
    for (std::thread& t : pool) t.join();
    // nothing of this call is left on the stream, also after an error
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e != hipSuccess ? e : (hipError_t)job.err.load();
  }

 private:
  // a filled slot and where its contents go
  static constexpr int kParts = 28;  // the populations' planes lie together
  struct Item {
    int slot = 0, parts = 0;
    struct {
      char* dst;
      size_t bytes;
    } part[kParts];
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
    if (e == hipSuccess) {
      const char* from = pin_ + (size_t)it.slot * kSlotBytes;
      for (int k = 0; k < it.parts; ++k) {
        memcpy(it.part[k].dst, from, it.part[k].bytes);
        from += it.part[k].bytes;
      }
    } else {
      job.err.store((int)e);
    }
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

  // At least n slots (1: a small read; kSlots: any other).  Asked for again
  // only where fewer had been refused.
  bool ensure_slots(int n) {
    if (slots_ >= n) return true;
    if (refused_ && n >= refused_) return false;
    void* p = nullptr;
    bool ok = hipHostMalloc(&p, kSlotBytes * n, hipHostMallocCoherent) == hipSuccess;
    while (ok && n > 1 && (int)ev_.size() < n) {
      hipEvent_t e;
      ok = hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem) == hipSuccess;
      if (ok) ev_.push_back(e);
    }
    if (!ok) {
      (void)hipGetLastError();
      if (p) (void)hipHostFree(p);
      refused_ = n;
      return false;
    }
    if (pin_) (void)hipHostFree(pin_);
    pin_ = (char*)p;
    slots_ = n;
    return true;
  }

  // Device workspace: as much as asked for up to kWorkBytes, or what a full
  // card still has of it; null when not even kMinWorkBytes can be had.
  void* work(size_t want, size_t* have) {
    want = std::min(std::max(want, kMinWorkBytes), kWorkBytes);
    if (work_bytes_ < want) {
      (void)release_work();
      for (work_bytes_ = want; hipMalloc(&work_, work_bytes_) != hipSuccess;) {
        (void)hipGetLastError();
        work_ = nullptr;
        if (work_bytes_ <= kMinWorkBytes) {
          work_bytes_ = 0;
          break;
        }
        work_bytes_ = std::max(work_bytes_ / 2, kMinWorkBytes);
      }
    }
    *have = work_bytes_;
    return work_;
  }

  char* pin_ = nullptr;
  int slots_ = 0, refused_ = 0;
  std::vector<hipEvent_t> ev_;
  void* work_ = nullptr;
  size_t work_bytes_ = 0;
};

// hipMalloc for every array of the library.  What the read-back keeps is given
// back before an allocation is refused.  The runtime holds a refusal for the next
// hipGetLastError, where it would be taken for a launch's: it is cleared here and
// reported by the caller alone.
template <typename T>
inline hipError_t gpu_malloc(T** p, size_t bytes, Readback* rb = nullptr) {
  hipError_t e = hipMalloc((void**)p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (rb && rb->release_work() && (e = hipMalloc((void**)p, bytes)) != hipSuccess) (void)hipGetLastError();
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

}  // namespace lbm

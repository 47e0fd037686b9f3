// kf_host_copy.hpp -- copies between a caller's pageable host arrays and one
// block of device memory, through pinned memory of the context.
//
// A copy of pageable memory costs ~8 us of the runtime's own staging however
// small it is, and a fit has up to 11 input and 24 output arrays: for 100
// tracks that was half of the call.  Large ones it stages at ~10 GB/s in one
// thread, and writing results into fresh memory takes the page faults there
// too.  Here the arrays are packed into one block per direction: small
// batches take one transfer each way, large ones chunks of kCopyChunk that a
// few threads fill or empty while others are on the bus.  Measured: a fit of
// 100 telescope tracks 495 -> 278 us, of 20 000 field-map tracks (16 MB in,
// 100 MB out) 15.5 -> 9.6 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

namespace kf {

constexpr size_t kCopyChunk = size_t{2} << 20;
constexpr int kCopyThreads = 8;
constexpr int kSlotsPerThread = 2;  // one on the bus, one being filled
// below this one transfer in the caller's thread
constexpr size_t kCopySingle = size_t{1} << 20;

// A host array's place in the device block.
struct CopyPiece {
  char* host;
  size_t off, bytes;
};

class HostCopy {
 public:
  // Pinned memory for a block of `total` bytes; false: there is none.
  bool reserve(size_t total) { return total == 0 || ensure(total) == hipSuccess; }

  // Packs the pieces and sends the block's first `total` bytes to `dev`.
  hipError_t upload(const CopyPiece* pieces, int count, char* dev, size_t total, int device,
                    hipStream_t s) {
    return run(total, device, [&](char* slot, hipEvent_t ev, size_t lo, size_t n) {
      // what the slot held last has left it
      hipError_t e = hipEventSynchronize(ev);
      if (e != hipSuccess) return e;
      forPieces(pieces, count, lo, n, [&](const CopyPiece& p, size_t a, size_t b) {
        std::memcpy(slot + (a - lo), p.host + (a - p.off), b - a);
      });
      e = hipMemcpyAsync(dev + lo, slot, n, hipMemcpyHostToDevice, s);
      return e != hipSuccess ? e : hipEventRecord(ev, s);
    });
  }

  // Brings the block back, after the work queued on `s`, and waits for it.
  hipError_t download(const CopyPiece* pieces, int count, const char* dev, size_t total,
                      int device, hipStream_t s) {
    if (total > kCopySingle) {
      // the threads start when there is something to copy
      if (const hipError_t e = hipStreamSynchronize(s)) return e;
    }
    return run(total, device, [&](char* slot, hipEvent_t ev, size_t lo, size_t n) {
      hipError_t e = hipMemcpyAsync(slot, dev + lo, n, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(ev, s);
      if (e == hipSuccess) e = hipEventSynchronize(ev);
      if (e != hipSuccess) return e;
      forPieces(pieces, count, lo, n, [&](const CopyPiece& p, size_t a, size_t b) {
        std::memcpy(p.host + (a - p.off), slot + (a - lo), b - a);
      });
      return hipSuccess;
    });
  }

  // Frees the pinned memory.
  void release() {
    settle();
    if (pinned_) (void)hipHostFree(pinned_);
    pinned_ = nullptr;
    bytes_ = 0;
    for (hipEvent_t& e : events_) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
  }

  // Whether `p` is ordinary host memory: anything else (pinned, managed)
  // the device copies by itself.
  static bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
      (void)hipGetLastError();
      return true;
    }
    return a.type == hipMemoryTypeUnregistered;
  }

 private:
  static constexpr int kSlots = kCopyThreads * kSlotsPerThread;
  char* pinned_ = nullptr;
  size_t bytes_ = 0;
  hipEvent_t events_[kSlots] = {};

  template <typename Fn>
  static void forPieces(const CopyPiece* pieces, int count, size_t lo, size_t n, Fn&& fn) {
    for (int i = 0; i < count; ++i) {
      const CopyPiece& p = pieces[i];
      const size_t a = std::max(lo, p.off), b = std::min(lo + n, p.off + p.bytes);
      if (a < b) fn(p, a, b);
    }
  }

  // Waits until nothing of the pinned memory is on the bus.
  void settle() {
    for (hipEvent_t e : events_)
      if (e) (void)hipEventSynchronize(e);
  }

  static int threadsFor(size_t total) {
    if (total <= kCopySingle) return 1;
    const int cpus = std::max(1u, std::thread::hardware_concurrency());
    return static_cast<int>(
        std::min<size_t>((total + kCopyChunk - 1) / kCopyChunk, std::min(kCopyThreads, cpus)));
  }

  hipError_t ensure(size_t total) {
    const int threads = threadsFor(total);
    const size_t need = threads == 1 && total <= kCopyChunk
                            ? (total + 65535) / 65536 * 65536
                            : kCopyChunk * kSlotsPerThread * threads;
    if (need > bytes_) {
      settle();
      if (pinned_) (void)hipHostFree(pinned_);
      pinned_ = nullptr;
      bytes_ = 0;
      void* p = nullptr;
      const hipError_t e = hipHostMalloc(&p, need, hipHostMallocDefault);
      if (e != hipSuccess) return e;
      pinned_ = static_cast<char*>(p);
      bytes_ = need;
    }
    for (hipEvent_t& ev : events_)
      if (!ev) {
        const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) return e;
      }
    return hipSuccess;
  }

  // chunk(slot, event, offset, bytes) for every chunk of the block: thread t
  // takes the chunks t, t + threads, ... with slots of its own.
  template <typename Chunk>
  hipError_t run(size_t total, int device, Chunk&& chunk) {
    if (total == 0) return hipSuccess;
    if (const hipError_t e = ensure(total)) return e;
    const int threads = threadsFor(total);
    const size_t step = threads == 1 ? std::min(bytes_, total) : kCopyChunk;
    std::atomic<int> error{hipSuccess};
    auto work = [&](int t) {
      hipError_t e = hipSetDevice(device);
      int k = 0;
      for (size_t lo = t * step; e == hipSuccess && lo < total && error == hipSuccess;
           lo += threads * step, ++k) {
        const int slot = threads == 1 ? 0 : t * kSlotsPerThread + k % kSlotsPerThread;
        e = chunk(pinned_ + slot * step, events_[slot], lo, std::min(step, total - lo));
      }
      if (e != hipSuccess) error = e;
    };
    std::thread pool[kCopyThreads];
    for (int t = 1; t < threads; ++t) {
      try {
        pool[t] = std::thread(work, t);
      } catch (const std::exception&) {
        work(t);  // no thread, or no memory for one: its share is done here
      }
    }
    work(0);
    for (std::thread& th : pool)
      if (th.joinable()) th.join();
    return static_cast<hipError_t>(error.load());
  }
};

}  // namespace kf

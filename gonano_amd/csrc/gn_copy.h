// gn_copy.h - large device-to-host copies (gradients, parameters, logits).
//
// hipMemcpy into pageable memory stages through one pinned buffer on one
// host thread, which also takes the page faults of a fresh destination:
// 10.4 GB/s for 80 MB of gradients (7.7 ms).  Here the caller queues pieces
// into a ring of pinned slots on its stream and up to THREADS - 1 helpers (and
// the caller, while the ring is full) copy arrived pieces out, so the link,
// the copies and the page faults overlap.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "gn_common.h"

namespace gn {

class HostCopy {
 public:
  struct Seg {
    void* host;
    const void* dev;
    size_t bytes;
  };
  static constexpr size_t PIECE = (size_t)1 << 20;  // a slot
  static constexpr int SLOTS = 12, THREADS = 7;

  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() { release(); }

  // Copies every segment (they do not overlap) behind the work queued on
  // `stream` and returns when all is in place.  Calls from several threads
  // take turns.
  void download(int device, hipStream_t stream, const std::vector<Seg>& segs) {
    std::lock_guard<std::mutex> lock(mu_);
    // pieces of at most PIECE bytes: large segments cut, small ones together
    std::vector<Seg> parts;
    std::vector<size_t> first;  // piece i: parts first[i] .. first[i + 1]
    size_t fill = PIECE;
    for (const Seg& s : segs)
      for (size_t o = 0; o < s.bytes;) {
        const size_t n = std::min(PIECE, s.bytes - o);
        if (fill + n > PIECE) {
          first.push_back(parts.size());
          fill = 0;
        }
        parts.push_back({(char*)s.host + o, (const char*)s.dev + o, n});
        fill += (n + 255) & ~(size_t)255;
        o += n;
      }
    const size_t n = first.size();
    if (n == 0) return;
    first.push_back(parts.size());
    // a ring of four slots for a few megabytes, of twelve from 48 MB: pinning
    // memory takes about 0.13 ms a megabyte, once per session
    const size_t slots = std::min<size_t>(n, std::max<size_t>(4, std::min<size_t>(SLOTS, n / 4)));
    reserve((int)slots);

    std::atomic<size_t> issued{0}, taken{0};
    std::atomic<size_t> freed[SLOTS];  // pieces a slot has passed on
    for (auto& f : freed) f.store(0);
    std::atomic<int> err{(int)hipSuccess};
    auto failed = [&] { return err.load() != (int)hipSuccess; };
    // copies piece j out of its slot once it has arrived
    auto drain = [&](size_t j) {
      while (issued.load(std::memory_order_acquire) <= j) {
        if (failed()) return;
        std::this_thread::yield();
      }
      const hipError_t e = hipEventSynchronize(done_[j % slots]);
      if (e != hipSuccess) {
        err.store((int)e);
        return;
      }
      const char* src = pin_ + (j % slots) * PIECE;
      for (size_t k = first[j]; k < first[j + 1]; k++) {
        std::memcpy(parts[k].host, src, parts[k].bytes);
        src += (parts[k].bytes + 255) & ~(size_t)255;
      }
      freed[j % slots].store(j / slots + 1, std::memory_order_release);
    };
    auto helper = [&] {
      const hipError_t e = hipSetDevice(device);
      if (e != hipSuccess) return;  // the others take its share
      for (size_t j; !failed() && (j = taken.fetch_add(1)) < n;) drain(j);
    };
    // Nothing between the first thread and the joins may throw: a thread (or
    // its memory) that cannot be had means fewer helpers, the caller takes
    // the rest.
    const size_t helpers = std::min<size_t>(THREADS, n) - 1;
    std::vector<std::thread> threads;
    threads.reserve(helpers);
    try {
      for (size_t l = 0; l < helpers; l++) threads.emplace_back(helper);
    } catch (const std::exception&) {
    }
    for (size_t i = 0; i < n && !failed();) {
      if (freed[i % slots].load(std::memory_order_acquire) == i / slots) {
        char* dst = pin_ + (i % slots) * PIECE;
        hipError_t e = hipSuccess;
        for (size_t k = first[i]; k < first[i + 1] && e == hipSuccess; k++) {
          e = hipMemcpyAsync(dst, parts[k].dev, parts[k].bytes, hipMemcpyDeviceToHost, stream);
          dst += (parts[k].bytes + 255) & ~(size_t)255;
        }
        if (e == hipSuccess) e = hipEventRecord(done_[i % slots], stream);
        if (e != hipSuccess) {
          err.store((int)e);
          break;
        }
        issued.store(++i, std::memory_order_release);
        continue;
      }
      // the ring is full: copy out a piece that is on its way, if one is untaken
      size_t j = taken.load();
      if (j < i && taken.compare_exchange_strong(j, j + 1)) drain(j);
      else std::this_thread::yield();
    }
    for (size_t j; !failed() && (j = taken.fetch_add(1)) < n;) drain(j);
    for (auto& t : threads) t.join();
    // nothing may still write the slots when the call returns
    const hipError_t e = hipStreamSynchronize(stream);
    GN_HIP((hipError_t)err.load());
    GN_HIP(e);
  }

  void release() {
    for (auto& d : done_) {
      if (d) (void)hipEventDestroy(d);
      d = nullptr;
    }
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
    slots_ = 0;
  }

 private:
  void reserve(int slots) {
    if (slots <= slots_) return;
    release();
    GN_HIP(hipHostMalloc((void**)&pin_, slots * PIECE, hipHostMallocDefault));
    for (int i = 0; i < slots; i++)
      GN_HIP(hipEventCreateWithFlags(&done_[i], hipEventDisableTiming));
    slots_ = slots;
  }
  std::mutex mu_;
  char* pin_ = nullptr;
  hipEvent_t done_[SLOTS] = {};
  int slots_ = 0;
};

}  // namespace gn

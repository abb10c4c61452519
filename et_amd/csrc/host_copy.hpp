// Device-to-host copies of long vectors into pageable memory.
//
// The runtime stages such a copy itself, one piece after the other on the calling
// thread: the 148 MB of (H2O)8's residual took 17 ms, most of it the first touch of
// a fresh array's pages.  Here pieces go to a ring of pinned buffers and a few
// threads move them on while the next ones are in flight: 6 ms.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "common.hpp"

namespace etg {

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() {
    for (hipEvent_t e : events_) (void)hipEventDestroy(e);
  }

  // Copies `bytes` from the device to `dst` after what is queued on `stream`; they are
  // there when the stream is next synchronised.  Short copies, and destinations the
  // runtime knows (pinned or device memory), go to it directly (9 MB: 0.1 ms saved
  // per copy against 1 ms for the first one's ring).
  void to_host(hipStream_t stream, void* dst, const void* src, size_t bytes) {
    if (bytes < kShortest || known_to_runtime(dst) || !prepare(kRing * piece_bytes(bytes))) {
      ETG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, stream));
      return;
    }
    const size_t piece = piece_bytes(bytes);
    const int n = int((bytes + piece - 1) / piece);
    std::atomic<int> next{0}, ready{0};
    std::atomic<bool> stop{false};
    std::vector<std::atomic<bool>> done(static_cast<size_t>(n));
    for (auto& d : done) d.store(false, std::memory_order_relaxed);
    auto length = [&](int i) { return std::min(piece, bytes - size_t(i) * piece); };
    auto slot = [&](int i) { return ring_.as<char>() + size_t(i % kRing) * piece; };
    auto move = [&] {
      for (int i; (i = next.fetch_add(1)) < n;) {
        while (ready.load(std::memory_order_acquire) <= i) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        std::memcpy(static_cast<char*>(dst) + size_t(i) * piece, slot(i), length(i));
        done[size_t(i)].store(true, std::memory_order_release);
      }
    };
    auto issue = [&](int i) {
      ETG_HIP(hipMemcpyAsync(slot(i), static_cast<const char*>(src) + size_t(i) * piece, length(i), hipMemcpyDeviceToHost,
                             stream));
      ETG_HIP(hipEventRecord(events_[size_t(i % kRing)], stream));
    };
    int issued = 0;
    for (; issued < std::min(n, kRing); ++issued) issue(issued);
    // the work queued before the copy may take seconds: the threads start when its first
    // piece is here (started before, they turned over in sched_yield: eight busy cores)
    ETG_HIP(hipEventSynchronize(events_[0]));
    struct Team {                         // joined on every way out
      std::atomic<bool>& stop;
      std::vector<std::thread> threads;
      ~Team() {
        stop.store(true);
        for (auto& t : threads) t.join();
      }
    } team{stop, {}};
    const int want = std::max(2, std::min({int(bytes / kPiece), kThreads, int(std::thread::hardware_concurrency())}));
    try {
      for (int t = 0; t < want; ++t) team.threads.emplace_back(move);
    } catch (const std::system_error&) {  // fewer threads, or none: the runtime's copy
    }
    if (team.threads.empty()) {
      ETG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream));
      return;
    }
    for (int i = 0; i < n; ++i) {
      ETG_HIP(hipEventSynchronize(events_[size_t(i % kRing)]));
      ready.store(i + 1, std::memory_order_release);
      // refill the slots that have been moved on; the next piece to wait for must be in flight
      while (issued < n && (done[size_t(issued - kRing)].load(std::memory_order_acquire) || issued == i + 1)) {
        while (!done[size_t(issued - kRing)].load(std::memory_order_acquire)) std::this_thread::yield();
        issue(issued++);
      }
    }
    for (int i = 0; i < n; ++i)
      while (!done[size_t(i)].load(std::memory_order_acquire)) std::this_thread::yield();
  }

 private:
  static constexpr size_t kShortest = size_t(16) << 20;
  static constexpr size_t kPiece = size_t(4) << 20;    // longest piece, one of the ring
  static constexpr int kRing = 8, kThreads = 8;

  static size_t piece_bytes(size_t bytes) {
    const size_t even = (bytes / (4 * kRing) + 4095) / 4096 * 4096;
    return std::max(size_t(256) << 10, std::min(kPiece, even));
  }
  static bool known_to_runtime(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return a.type != hipMemoryTypeUnregistered;
  }
  bool prepare(size_t ring_bytes) {
    if (refused_) return false;
    try {
      ring_.resize_host(ring_bytes);
      while (events_.size() < size_t(kRing)) {
        hipEvent_t e;
        ETG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        events_.push_back(e);
      }
    } catch (const Error&) {
      (void)hipGetLastError();
      refused_ = true;
      return false;
    }
    return true;
  }

  DeviceBuffer ring_;                       // pinned host memory
  std::vector<hipEvent_t> events_;
  bool refused_ = false;
};

}  // namespace etg

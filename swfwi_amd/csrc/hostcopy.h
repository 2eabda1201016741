// Large copies between device arrays and the caller's pageable memory, and
// that memory's first touch.
#pragma once
#include <atomic>
#include <cstddef>
#include <thread>
#include <vector>

#include "device.h"

namespace swfwi {

struct HostSpan {
  void* host;
  void* dev;
  size_t bytes;
};

// Pinned staging of one handle for its large copies: pieces of 2 MB go
// through pinned slots, each worker (the caller and three threads that live
// for the call) with two slots, one on its way while the other is copied to
// or from the caller's memory.  The runtime's own pageable copy is one thread
// copying next to the transfer: 80 MB down 5.0 ms that way and 2.2 with the
// workers (into pages that exist), up 3.0 and 2.2.  A total below
// kHostCopyFrom goes to the runtime: 24 MB are 1.56 -> 0.76 ms down and
// 0.84 -> 0.72 up, and the gain up ends at 16 MB (0.46 ms).  Memory that the
// runtime knows goes to it as well: it transfers pinned memory without a copy
// (77 MB 1.43 ms up and 1.44 down, in pieces 2.13 and 2.13).
// 16 MB of pinned memory, allocated on the first large copy (0.5 ms) and
// given back with the handle; where they cannot be had the runtime copies.
constexpr size_t kHostCopyFrom = 16u << 20;
class HostLane {
 public:
  HostLane() = default;
  ~HostLane();
  HostLane(const HostLane&) = delete;
  HostLane& operator=(const HostLane&) = delete;
  // After the work queued on s; the data is in place on return.
  void down(const std::vector<HostSpan>& spans, hipStream_t s) { run(spans, s, true); }
  // Before the work queued on s after the call; the caller's memory is free
  // on return.
  void up(const std::vector<HostSpan>& spans, hipStream_t s) { run(spans, s, false); }

 private:
  static constexpr int kWorkers = 4;
  static constexpr size_t kPiece = 2u << 20;
  bool slots();
  void run(const std::vector<HostSpan>& spans, hipStream_t s, bool down);
  char* pin_ = nullptr;
  hipEvent_t done_[2 * kWorkers] = {};
};

// First touch of memory that a run's results will go to, by threads next to
// the run: a fresh allocation's pages cost 3.5 to 11 ms for 88 MB, which the
// copy would otherwise pay after the run.  The bytes keep their values.
// Nothing below kHostCopyFrom or for memory that the runtime knows, whose pages
// exist; the destructor waits.
class PageIn {
 public:
  PageIn(void* p, size_t bytes);
  ~PageIn();
  PageIn(const PageIn&) = delete;
  PageIn& operator=(const PageIn&) = delete;
  void wait();

 private:
  std::atomic<bool> stop_{false};
  std::vector<std::thread> threads_;
};

}  // namespace swfwi

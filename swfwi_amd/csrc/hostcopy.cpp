#include "hostcopy.h"

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>

namespace swfwi {

namespace {
// Memory the runtime knows (pinned, managed or a device's): it copies that
// directly, and the host may not be able to touch it at all.
bool known_to_runtime(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // ordinary memory
  return false;
}
}  // namespace

HostLane::~HostLane() {
  for (hipEvent_t e : done_)
    if (e) (void)hipEventDestroy(e);
  if (pin_) (void)hipHostFree(pin_);
}

// whether the pinned slots are there; without them the runtime copies
bool HostLane::slots() {
  if (!pin_ && hipHostMalloc((void**)&pin_, 2 * kWorkers * kPiece, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    pin_ = nullptr;
  }
  return pin_ != nullptr;
}

void HostLane::run(const std::vector<HostSpan>& spans, hipStream_t s, bool down) {
  size_t total = 0;
  for (const HostSpan& p : spans) total += p.bytes;
  const bool known = total > 0 && known_to_runtime(spans.front().host);
  if (total < kHostCopyFrom || known || !slots()) {
    for (const HostSpan& p : spans) {
      if (down)
        SWFWI_HIP(hipMemcpyAsync(p.host, p.dev, p.bytes, hipMemcpyDeviceToHost, s));
      else
        SWFWI_HIP(hipMemcpyAsync(p.dev, p.host, p.bytes, hipMemcpyHostToDevice, s));
    }
    if (down || known) SWFWI_HIP(hipStreamSynchronize(s));
    return;
  }
  for (hipEvent_t& e : done_)
    if (!e) SWFWI_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  int device = 0;
  SWFWI_HIP(hipGetDevice(&device));
  std::vector<HostSpan> pieces;
  for (const HostSpan& p : spans)
    for (size_t o = 0; o < p.bytes; o += kPiece)
      pieces.push_back({(char*)p.host + o, (char*)p.dev + o, std::min(kPiece, p.bytes - o)});
  std::atomic<size_t> next{0};
  std::mutex mu;
  std::exception_ptr error;
  auto worker = [&](int k) {
    try {
      SWFWI_HIP(hipSetDevice(device));
      char* slot[2] = {pin_ + 2 * k * kPiece, pin_ + (2 * k + 1) * kPiece};
      hipEvent_t* done = done_ + 2 * k;
      auto take = [&]() -> const HostSpan* {
        const size_t i = next++;
        return i < pieces.size() ? &pieces[i] : nullptr;
      };
      if (down) {
        auto start = [&](const HostSpan* p, int q) {
          if (!p) return;
          SWFWI_HIP(hipMemcpyAsync(slot[q], p->dev, p->bytes, hipMemcpyDeviceToHost, s));
          SWFWI_HIP(hipEventRecord(done[q], s));
        };
        int q = 0;
        const HostSpan* cur = take();
        start(cur, q);
        for (; cur; q ^= 1) {
          const HostSpan* nxt = take();
          start(nxt, q ^ 1);
          SWFWI_HIP(hipEventSynchronize(done[q]));
          std::memcpy(cur->host, slot[q], cur->bytes);
          cur = nxt;
        }
      } else {
        bool used[2] = {false, false};
        int q = 0;
        for (const HostSpan* p; (p = take()); q ^= 1) {
          if (used[q]) SWFWI_HIP(hipEventSynchronize(done[q]));
          std::memcpy(slot[q], p->host, p->bytes);
          SWFWI_HIP(hipMemcpyAsync(p->dev, slot[q], p->bytes, hipMemcpyHostToDevice, s));
          SWFWI_HIP(hipEventRecord(done[q], s));
          used[q] = true;
        }
        for (q = 0; q < 2; q++)
          if (used[q]) SWFWI_HIP(hipEventSynchronize(done[q]));
      }
    } catch (...) {
      next = pieces.size();  // the others stop
      std::lock_guard<std::mutex> l(mu);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> threads;
  threads.reserve(kWorkers);
  const int extra = std::min<int>(kWorkers, std::max(1u, std::thread::hardware_concurrency())) - 1;
  for (int k = 1; k <= extra; k++) {
    try {
      threads.emplace_back(worker, k);
    } catch (const std::exception&) {
      break;  // no more threads to be had: those there are do it
    }
  }
  worker(0);
  for (std::thread& t : threads) t.join();
  if (error) {
    (void)hipStreamSynchronize(s);  // no copy may use a slot after the call
    std::rethrow_exception(error);
  }
}

PageIn::PageIn(void* p, size_t bytes) {
  if (!p || bytes < kHostCopyFrom || known_to_runtime(p)) return;
  constexpr size_t kPage = 4096;
  const int n = std::min<int>(4, std::max(1u, std::thread::hardware_concurrency()));
  char* base = (char*)p;
  try {
    threads_.reserve(n);
    for (int k = 0; k < n; k++) {
      char *a = base + bytes / n * k, *b = k + 1 < n ? base + bytes / n * (k + 1) : base + bytes;
      threads_.emplace_back([this, a, b] {
        for (char* q = a; q < b && !stop_.load(std::memory_order_relaxed); q += kPage)
          __atomic_fetch_or(q, (char)0, __ATOMIC_RELAXED);
      });
    }
  } catch (const std::exception&) {
    // no more threads to be had: the copy touches the rest
  }
}

void PageIn::wait() {
  for (std::thread& t : threads_) t.join();
  threads_.clear();
}

PageIn::~PageIn() {
  stop_ = true;
  wait();
}

}  // namespace swfwi

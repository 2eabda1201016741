// The large host copies against a runtime of this file's own: device memory is
// host memory, every call is counted, and allocations can be made to fail.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>

#include "hostcopy.h"

static bool g_known = false, g_pin_fails = false;
static int g_copies = 0, g_syncs = 0;
static size_t g_largest = 0, g_total = 0;

extern "C" {
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  if (!g_known) return hipErrorInvalidValue;
  a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  __atomic_add_fetch(&g_copies, 1, __ATOMIC_SEQ_CST);
  __atomic_add_fetch(&g_total, n, __ATOMIC_SEQ_CST);
  if (n > g_largest) g_largest = n;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_pin_fails) return hipErrorOutOfMemory;
  return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { g_syncs++; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "test"; }
}

static int g_news = 0;  // the g_news-th allocation from here on fails (0: none)
void* operator new(size_t n) {
  if (g_news > 0 && __atomic_sub_fetch(&g_news, 1, __ATOMIC_SEQ_CST) == 0) throw std::bad_alloc();
  void* p = std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

using namespace swfwi;

static bool moves(HostLane& lane, bool down, size_t n) {
  char *h = (char*)std::malloc(n), *d = (char*)std::malloc(n);
  for (size_t i = 0; i < n; i += 511) d[i] = (char)(i / 511), h[i] = (char)(i / 511 + 1);
  std::vector<HostSpan> v{{h, d, n / 3}, {h + n / 3, d + n / 3, n - n / 3}};
  if (down)
    lane.down(v, nullptr);
  else
    lane.up(v, nullptr);
  bool same = true;
  for (size_t i = 0; i < n; i += 511) same = same && h[i] == d[i] && h[i] == (char)(i / 511 + (down ? 0 : 1));
  std::free(h);
  std::free(d);
  return same;
}

int main(int, char** argv) {
  const std::string what = argv[1];
  const size_t n = (24u << 20) + 12345;
  for (bool down : {true, false}) {
    g_copies = g_syncs = 0;
    g_largest = g_total = 0;
    if (what == "pageable" || what == "known" || what == "no_pin") {
      g_known = what == "known";
      g_pin_fails = what == "no_pin";
      HostLane lane;
      if (!moves(lane, down, n)) return 1;
      std::printf("%d copies, largest %zu, total %zu, syncs %d\n", g_copies, g_largest, g_total, g_syncs);
      if (g_total != n || (what == "pageable" ? g_largest != 2u << 20 : g_copies != 2)) return 2;
      if (what == "known" && g_syncs != 1) return 3;  // the caller's memory is its own again
    } else {
      HostLane lane;
      if (!moves(lane, down, n)) return 4;  // the slots exist
      for (int k = 1; k < 40; k++) {
        g_news = k;
        try {
          if (!moves(lane, down, n)) return 5;
        } catch (const std::bad_alloc&) {
        }
        g_news = k;
        try {
          char* p = (char*)std::malloc(n);
          { PageIn in(p, n); }
          std::free(p);
        } catch (const std::bad_alloc&) {
          return 6;  // it only helps
        }
        g_news = 0;
      }
    }
  }
  if (what == "known") {  // memory the host may not touch is not paged in
    g_known = true;
    PageIn in((void*)64, n);
  }
  return 0;
}

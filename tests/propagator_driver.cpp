// The propagator's host side against a runtime and launchers of this file's
// own: nothing runs, what is launched is counted, a resident run can be told to
// find the chip shared, and allocations can be made to fail.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>

#include "propagator.h"

using namespace swfwi;

static int g_fwd = 0, g_bwd = 0, g_march = 0, g_resident[2] = {0, 0};
static bool g_shared[2] = {false, false}, g_no_pinned = false;
static int g_memory = 1 << 30;  // allocations that succeed
static long long g_limit = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (g_memory-- <= 0) return hipErrorOutOfMemory;
  return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_no_pinned) return hipErrorOutOfMemory;
  return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "test"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free((void*)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = nullptr; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

namespace swfwi {
int tile_count_x(int nx, int tile_x) { return (nx - 2 * kHalo + tile_x - 1) / tile_x; }
void launch_fill(float*, long long, float, hipStream_t) {}
void launch_fill_u32(unsigned*, long long, unsigned, hipStream_t) {}
void launch_point_inject(float*, long long, const Inject&, int, int, hipStream_t) {}
void launch_fwd_step(const FwdStepArgs&, int, bool, int, hipStream_t, int) { g_fwd++; }
void launch_bwd_step(const BwdStepArgs&, int, int, hipStream_t, int) { g_bwd++; }
void launch_fwd_march(const FwdStepArgs&, const MarchMap&, int, int, hipStream_t) { g_march++; }
int resident_cus() { return 256; }
int resident_per_cu(bool backward, int, int) { return backward ? 1 : 2; }
static void resident(int kind, const ResComm& x) {
  g_resident[kind]++;
  g_limit = x.limit;
  if (!x.buf || !x.abort_dev || !x.abort_host) std::abort();
  if (g_shared[kind]) *x.abort_host = 1;
}
void launch_resident_fwd(const ResFwdArgs& a, int, hipStream_t) { resident(0, a.x); }
void launch_resident_bwd(const ResBwdArgs& a, int, hipStream_t) { resident(1, a.x); }
}  // namespace swfwi

struct Size {
  int ux, uz, nt = 350, receivers = 1;  // update region; dt = 2 ms: imaging from step 151 on
};
struct Run {
  Propagator p;
  Fields w;
  std::vector<float> v;  // stands in for every array of the caller's
  int nt;
  static Geometry geometry(const Size& s) {
    Geometry g;
    g.nx = s.ux - 40, g.nz = s.uz - 20, g.nb = 20, g.dt = 0.002f, g.dx = 20, g.fm = 12, g.nt = s.nt;
    g.sx = {3}, g.sz = {1}, g.gx.assign(s.receivers, 9), g.gz.assign(s.receivers, 1);
    return g;
  }
  explicit Run(const Size& s, int precision = kExact) : p(geometry(s), precision), v(64), nt(s.nt) {}
  explicit Run(int nt_, bool crowded = false) : Run(Size{341, 221, nt_, crowded ? 700 : 1}) {}
  Propagator::Sources src() { return Propagator::Sources{v.data(), 1, 0, nullptr, nullptr}; }
  // launches of the per-step kernels (trials included), resident launches; the run's route
  int forward(int E, bool band) {
    g_fwd = g_bwd = g_march = g_resident[0] = g_resident[1] = 0;
    p.forward(E, v.data(), 0, src(), nullptr, band ? v.data() : nullptr, w);
    return p.last_run[0].route;
  }
  int backward(int E) {
    g_fwd = g_bwd = g_resident[0] = g_resident[1] = 0;
    p.backward(E, v.data(), 0, src(), v.data(), 0, v.data(), v.data(), p.geo().npts(), w);
    return p.last_run[1].route;
  }
};

#define EXPECT(c) do { if (!(c)) { std::printf("line %d: %s (fwd %d bwd %d)\n", __LINE__, #c, g_fwd, g_bwd); return 1; } } while (0)
constexpr int kTrial = 3 * kNumWidths * 8;  // launches of one kernel's width trials

static int tuner() {
  const int nt = 170;
  Run fresh(nt), used(nt);
  fresh.p.set_resident(0, 5e5);
  EXPECT(fresh.forward(8, true) == Propagator::kPerStep);
  EXPECT(g_fwd == nt + kTrial && g_bwd == kTrial);
  EXPECT(used.forward(8, true) == Propagator::kResident);
  EXPECT(g_fwd == 0 && g_bwd == 0 && g_resident[0] == 1);
  EXPECT(used.p.tile_choice_cached(0, 8) > 0 && used.p.tile_choice_cached(1, 8) > 0);
  used.p.set_resident(0, 5e5);
  EXPECT(used.forward(8, true) == Propagator::kPerStep);
  EXPECT(g_fwd == nt + kTrial && g_bwd == kTrial);  // as a new handle's
  EXPECT(used.forward(8, true) == Propagator::kPerStep);
  EXPECT(g_fwd == nt && g_bwd == 0);
  used.p.set_tuning(false);
  EXPECT(used.forward(8, true) == Propagator::kPerStep && g_fwd == nt && g_bwd == 0);
  return 0;
}

static int backward_trials() {
  const int nt = 170;
  Run r(nt);
  r.p.set_resident(0, 5e5);
  EXPECT(r.forward(30, false) == Propagator::kPerStep && g_fwd == nt + kTrial && g_bwd == 0);  // nothing follows
  EXPECT(r.p.tile_choice_cached(1, 30) > 0);
  EXPECT(r.forward(30, true) == Propagator::kPerStep && g_fwd == nt && g_bwd == kTrial);
  EXPECT(r.backward(30) == Propagator::kPerStep && r.p.last_run[1].width == r.p.tile_choice_cached(1, 30));
  Run s(350);  // 34 entries: the forward a launch a step, the backward resident in parts
  EXPECT(s.forward(34, true) == Propagator::kPerStep && g_fwd == 350 + kTrial && g_bwd == 0);
  EXPECT(s.backward(34) == Propagator::kResident && g_resident[1] >= 2 && g_bwd == 0);
  Run c(nt, true);  // more receivers at a place than a resident tile takes
  EXPECT(c.forward(8, true) == Propagator::kPerStep && g_bwd == kTrial && g_resident[0] == 0);
  EXPECT(c.backward(8) == Propagator::kPerStep);
  return 0;
}

static int no_memory() {
  for (int left = -1; left < 16; left++) {  // the allocation that fails (-1: pinned memory)
    Run r(170);
    r.p.set_resident(0, 5e5);
    r.forward(8, true);  // the fields and lists exist
    r.backward(8);
    r.p.set_resident(-1, 5e5);
    if (left >= 0) g_memory = left;
    g_no_pinned = left < 0;
    const int f = r.forward(8, true), b = r.backward(8);
    if (left <= 0) EXPECT(f == Propagator::kPerStep && b == Propagator::kPerStep);
    if (left == 15) EXPECT(f == Propagator::kResident && b == Propagator::kResident && g_memory > 0);
    EXPECT(r.p.gave_up == 0);
    g_memory = 1 << 30;
    g_no_pinned = false;
    EXPECT(r.forward(8, true) == Propagator::kResident && r.backward(8) == Propagator::kResident);
  }
  return 0;
}

// runs of a kind until the next one that tries the resident loop
static int runs_until_a_try(Run& r, int kind) {
  for (int k = 1; k < 20000; k++) {
    r.forward(8, true);
    const bool forward_tried = g_resident[0] > 0;
    if (kind == 0 && forward_tried) return k;
    r.backward(8);
    if (kind == 1 && g_resident[1] > 0) return k;
  }
  return -1;
}

static int shared_chip() {
  for (int kind = 0; kind < 2; kind++) {
    Run r(170);
    g_shared[kind] = true;
    EXPECT(runs_until_a_try(r, kind) == 1 && r.p.last_run[kind].route == Propagator::kPerStep && r.p.gave_up == 1);
    long long last = 64;
    EXPECT(runs_until_a_try(r, kind) == last && r.p.gave_up == 2);
    for (int k = 0; k < 8; k++) {  // rarer each time, up to a limit
      const long long n = runs_until_a_try(r, kind);
      EXPECT(n == (2 * last < 4096 ? 2 * last : 4096));
      last = n;
    }
    EXPECT(last == 4096 && r.p.gave_up == 10);
    g_shared[kind] = false;  // the chip is free again
    EXPECT(runs_until_a_try(r, kind) == 4096 && r.p.last_run[kind].route == Propagator::kResident);
    EXPECT(runs_until_a_try(r, kind) == 1 && r.p.last_run[kind].route == Propagator::kResident);
    g_shared[kind] = true;
    EXPECT(runs_until_a_try(r, kind) == 1 && r.p.gave_up == 11 && runs_until_a_try(r, kind) == 64);
    r.p.set_resident(-1, 5e5);  // asked for: at once
    EXPECT(runs_until_a_try(r, kind) == 1);
    g_shared[kind] = false;
  }
  return 0;
}

static int wait_limit() {
  Run r(170);
  for (double bad : {-1.0, (double)NAN, (double)INFINITY}) {
    bool refused = false;
    try {
      r.p.set_resident(1, bad);
    } catch (const Error& e) {
      refused = e.code == kErrArg;
    }
    EXPECT(refused);
  }
  for (double us : {0.0, 5e5, 1e7, 1e8, 1e300}) {
    r.p.set_resident(1, us);
    EXPECT(r.forward(8, true) == Propagator::kResident);
    EXPECT(g_limit == (long long)((us < 1e7 ? us : 1e7) * 100));  // ticks of the clock above
  }
  return 0;
}

static int few_steps() {
  for (int nt = 1; nt < 8; nt++) {
    Run r(nt);
    EXPECT(r.forward(1, false) == (nt < 5 ? Propagator::kPerStep : Propagator::kResident));
    r.p.set_resident(1, 5e5);
    EXPECT(r.forward(1, false) == (nt < 2 ? Propagator::kPerStep : Propagator::kResident));
  }
  return 0;
}

// Batches measured both ways (launches a run, 0: a launch a step), 200 backward
// iterations; the region's last tiles of 62 z are nearly empty in the first ones.
static int parts() {
  struct {
    Size s;
    int E, fwd, bwd;
  } const cases[] = {
      {{340, 63}, 75, 0, 0},   // backward 19.5 us a launch a step, 23.2 in 5 parts
      {{700, 63}, 30, 0, 0},   // forward 8.9, 9.7 in 2; backward 16.8, 18.8 in 4
      {{700, 125}, 19, 0, 0},  // forward 9.7, 10.2 in 2; backward 17.3, 19.1 in 4
      {{340, 125}, 54, 0, 0},  // backward 22.7, 27.8 in 5
      {{340, 125}, 22, 2, 2},  // backward 12.4, 9.8 in 2
      {{700, 187}, 22, 0, 0},  // backward 24.5, 28.6 in 6
      {{341, 221}, 16, 1, 2},  // backward 13.7, 10.4 in 2
      {{341, 221}, 22, 2, 3},  // forward 10.0, 6.7 in 2; backward 17.9, 15.5 in 3
      {{981, 331}, 8, 2, 4},   // forward 11.9, 10.1 in 2; backward 23.7, 20.3 in 4
      {{160, 110}, 100, 2, -1},  // forward 11.0, 6.8 in 2
  };
  for (const auto& c : cases) {
    Run r(c.s);
    r.p.set_tuning(false);
    const int f = r.forward(c.E, true), fl = r.p.last_run[0].launches;
    r.backward(c.E);
    const bool rb = r.p.last_run[1].route == Propagator::kResident;
    std::printf("%d x %d, %d entries: forward route %d, %d launches; backward route %d, %d\n", c.s.ux, c.s.uz, c.E, f,
                fl, r.p.last_run[1].route, r.p.last_run[1].launches);
    EXPECT(c.fwd ? f == Propagator::kResident && fl == c.fwd : f != Propagator::kResident);
    if (c.bwd >= 0) EXPECT(c.bwd ? rb && r.p.last_run[1].launches == c.bwd : !rb);
  }
  // one launch of 15 rows in FP32: 7.6 us against 7.0
  Run wide(Size{340, 63}, kFp32);
  EXPECT(wide.forward(39, true) == Propagator::kPerStep);
  // a launch of each part has to pay: 20 backward iterations in place of 200
  // (31.4 us in 3 parts against 28.9; with 200 iterations 19.1 against 19.4)
  Run few(Size{340, 331, 170}), many(Size{340, 331, 350});
  few.forward(16, true), many.forward(16, true);
  EXPECT(few.backward(16) == Propagator::kPerStep && many.backward(16) == Propagator::kResident);
  // 2 to 4 entries run side by side where their tiles are wide: 331 z, 4 of 700 x 4.9 us against 5.1
  Run four(Size{700, 331}), three(Size{700, 331});
  EXPECT(four.forward(4, false) == Propagator::kSideBySide && three.forward(3, false) == Propagator::kResident);
  EXPECT(four.forward(4, true) == Propagator::kResident);  // (with a band there are no streams to take)
  return 0;
}

int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "tuner") return tuner();
  if (what == "backward_trials") return backward_trials();
  if (what == "no_memory") return no_memory();
  if (what == "shared_chip") return shared_chip();
  if (what == "wait_limit") return wait_limit();
  if (what == "few_steps") return few_steps();
  if (what == "parts") return parts();
  return 2;
}

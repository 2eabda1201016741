// Host side of the resident time loop: which runs take it, the tiles and point
// lists of a run, its exchange buffer, and the launch under the device's lock.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>

#include "batch.h"
#include "propagator.h"

namespace swfwi {

namespace {

// One resident run at a time onto a device: two of them could each hold part
// of the chip and wait for blocks that cannot start.
constexpr int kMaxDevices = 64;
std::mutex& device_lock(int dev) {
  static std::mutex mu[kMaxDevices];
  return mu[dev >= 0 && dev < kMaxDevices ? dev : 0];
}

// Whether the buffers that `get` asks for could be had: without them the
// per-step kernels run.
template <class F>
bool had(F&& get) {
  try {
    get();
    return true;
  } catch (const Error& e) {
    if (e.code != kErrHip) throw;
    (void)hipGetLastError();
    return false;
  }
}

struct HostPoints {
  std::vector<int> ptr;
  std::vector<int2> items;
  int most = 0;
};

HostPoints bucket(const std::vector<long long>& idx, int ld, const ResTiles& t) {
  std::vector<std::vector<int2>> lists(t.n());
  for (size_t i = 0; i < idx.size(); i++) {
    const int ix = (int)(idx[i] / ld) - kHalo, iz = (int)(idx[i] % ld) - kHalo;
    const int tx = ix / t.w, tz = iz / t.h;
    lists[(size_t)tx * t.ntz + tz].push_back(make_int2(((ix - tx * t.w) << 6) | (iz - tz * t.h + 1), (int)i));
  }
  HostPoints h;
  h.ptr.push_back(0);
  for (const auto& l : lists) {
    h.items.insert(h.items.end(), l.begin(), l.end());
    h.ptr.push_back((int)h.items.size());
    h.most = std::max(h.most, (int)l.size());
  }
  return h;
}

}  // namespace

void Propagator::set_resident(int mode, double wait_us) {
  if (mode < -1 || mode > 1) fail(kErrArg, "resident mode must be -1 (by rule), 0 or 1");
  if (!(wait_us >= 0) || std::isinf(wait_us)) fail(kErrArg, "the resident wait limit must be finite and not negative");
  resident_ = mode;
  res_wait_us_ = std::min(wait_us, kResWaitMostUs);
  res_rest_ = 0;
  res_pause_[0] = res_pause_[1] = kResPause;
}

bool Propagator::res_twice(int rows) {
  if (rows > kResTwiceRows) return false;
  int& known = res_twice_[prec_][rows];
  if (!known) known = resident_per_cu(false, prec_, rows * kResWaves) >= 2 ? 1 : -1;
  return known == 1;
}

// A batch too large for the chip, or one whose tiles would be very wide, is
// faster as a few resident launches one after the other, each with
// tiles of a size that costs least a row.  Measured, microseconds a step.
// Forward, a launch a step -> in parts: 201x301 E=22 10.0 -> 6.7, E=26 10.7 ->
// 9.1, E=33 12.1 -> 10.1, 301x921 E=8 11.9 -> 10.1, 90x120 E=80 10.4 -> 7.9,
// E=100 11.0 -> 6.8; E=20 as one launch of 16 rows 8.65 -> 7.6 (of 14 rows, 10
// entries of 250x500, 7.07 -> 7.3).  Parts of 9 rows a wave lose: 301x921 E=5
// 9.4 -> 10.0 (in three of 3 rows 8.35).  Three parts pay at 4 rows, in exact
// mode also at 3 (250x500 E=12 10.0 -> 9.7, in FP32 9.35 -> 10.15); 301x921
// E=12 in FP32, 6 rows, 13.6 -> 14.3.  Three of 5 rows are left to the per-step
// kernels: whole calls of 201x301 E=38 13.8 -> 14.2 in exact mode, 12.9 -> 12.6 in
// FP32, 301x921 E=9 13.1 -> 13.2, but 90x120 E=160 16.3 -> 13.5.  Backward: 201x301 E=13 12.6 -> 9.2,
// E=16 13.7 -> 10.4, E=22 17.9 -> 15.5, 301x921 E=6 19.1 -> 15.5, 90x120
// E=100 20.6 -> 18.4; one launch of 10 rows 12.4 -> 9.2 (90x120 E=60), of 9
// rows the same, of 8 rows 7.8 -> 8.1 (201x301 E=10).
// More parts pay backward only: 201x301 E=32 24.8 -> 20.9, E=60 46.9 -> 43.5,
// 301x921 E=8 23.7 -> 20.3, E=13 35.2 -> 35.3, E=16 43.6 -> 40.6, 90x120 E=200
// 41.9 -> 31.3; forward the strip walk has caught up (201x301 E=40: 14.0).
// All of these fill their tiles of 62 z well; where the last tile of a column is
// nearly empty (63, 125, 187 z) parts lose: backward 700x63 E=54 25.7 -> 33.2,
// 340x125 E=75 30.1 -> 40.3, 700x187 E=22 24.5 -> 28.6, forward 700x63 E=30 8.9 ->
// 9.7, 340x125 E=39 9.8 -> 10.5.  So parts are taken where their time, by the
// tables below, is under the per-step kernels': of 1518 backward and 1315 forward
// batches (62 to 331 z, 130 to 1000 x, 2 to 90 entries, both modes) none that is
// taken was slower by more than 2%, but one (130x63 E=90, forward 7.3 -> 7.8).
// 2 to 4 forward entries without a band could run side by side on streams, with
// a launch a step, and do where their tiles are wide: 501x1501 E=2 7.0 against 7.3
// us a step, 1000x331 E=3 (9 rows) 4.9 against 5.0, E=4 (6 rows, two blocks a CU)
// 5.0 against 5.2, 700x331 E=4 (9 rows) 4.9 against 5.1, E=3 (7 rows) 4.7 against
// 3.9.
int Propagator::plan_parts(int kind, int E, bool band, ResTiles& t) {
  const auto rows = [](const ResTiles& r) { return (r.w + kResWaves - 1) / kResWaves; };
  const bool one = plan_resident(kind, E, t);
  if (resident_ == 1) return one ? 1 : 0;
  if (one && kind == 0 && side_by_side(E, band) && rows(t) > (two_a_cu(kind, E, t) ? kResLanesRows2 : kResLanesRows)) return 0;
  if (one && rows(t) < (kind == 1 ? kResWideBwd : kResWideFwd)) return 1;
  const double margin = kind == 1 ? 1.0 : 0.92;
  for (int n = 2; n <= (kind == 1 ? kResMaxPartsBwd : kResMaxPartsFwd) && n < E; n++) {
    ResTiles p;
    if (!plan_resident(kind, (E + n - 1) / n, p)) continue;
    const int r = rows(p);
    if (kind == 1 || n == 2 ? r > kResPartRows : r != 4 && (prec_ != kExact || r != 3)) continue;
    const double steps = kind == 1 ? bwd_iters_ : g_.nt;
    if (n * (part_us(kind, (E + n - 1) / n, p) + kResPartUs / steps) > margin * step_us(kind, E)) continue;
    t = p;
    return n;
  }
  // one launch of very wide tiles (forward 15 or 16 rows, backward 10)
  return one && (kind == 1 || kResWideUs[prec_] < margin * step_us(kind, E)) ? 1 : 0;
}

// Microseconds a step of a resident launch by its rows a wave, the medians of the
// measurements above (each within 10%): backward, forward with one block a CU
// and with two.
double Propagator::part_us(int kind, int E, const ResTiles& t) const {
  static const double us[2][3][kResPartRows] = {
      {{2.7, 2.9, 3.3, 3.9, 4.4, 4.9, 5.7}, {2.0, 2.2, 2.6, 2.9, 3.6, 3.8, 4.0}, {2.4, 2.7, 3.0, 3.4, 4.4, 5.1, 5.1}},
      {{2.6, 2.8, 3.1, 3.3, 4.1, 4.5, 4.9}, {1.9, 2.1, 2.5, 2.8, 3.3, 3.5, 3.7}, {2.4, 2.7, 3.1, 3.5, 4.0, 4.7, 4.7}}};
  const int rows = std::min((t.w + kResWaves - 1) / kResWaves, kResPartRows);
  return us[prec_][kind == 1 ? 0 : two_a_cu(kind, E, t) ? 2 : 1][rows - 1];
}
// ... and of the per-step kernels: a launch, the columns of 64-z tiles, and the
// points of the boundary band and sponge (fitted to the same batches, within 10%
// from 600 tiles of 64 x 16 on).
double Propagator::step_us(int kind, int E) const {
  static const double fit[2][2][3] = {{{4.54, 0.00217, 0.0061}, {5.19, 0.00546, 0.0151}},
                                      {{4.51, 0.00180, 0.0058}, {4.84, 0.00505, 0.0155}}};
  const int ux = g_.nxpad - 2 * kHalo, uz = g_.nzpad - 2 * kHalo;
  const double* f = fit[prec_][kind];
  return f[0] + E * (f[1] * g_.ntz * ux / 16 + f[2] * (2 * uz + ux) / 100);
}

bool Propagator::runs_resident(int kind, int E, bool band) {
  ResTiles t;
  if (plan_parts(kind, E, band, t) < 1) return false;
  const ResLayout* l = res_layout(t);
  return l && l->fits;
}

bool Propagator::plan_resident(int kind, int E, ResTiles& t) {
  if (resident_ == 0 || tile_override_ || (kind == 1 && bwd_split_ >= 0) || g_.nt < 2) return false;
  const int most = kind == 1 ? kResMaxWidthBwd : kResMaxWidthFwd;
  int& cap = res_cap_[kind][prec_];
  if (cap < 0) {  // every width's kernel fits at least one block a CU
    cap = resident_cus();
    for (int w = kResWaves; w <= most; w += kResWaves)
      if (resident_per_cu(kind == 1, prec_, w) < 1) cap = 0;
  }
  const int ux = g_.nxpad - 2 * kHalo, uz = g_.nzpad - 2 * kHalo;
  t.ntz = (uz + kResTileZ - 1) / kResTileZ;
  t.h = (uz + t.ntz - 1) / t.ntz;
  t.ntz = (uz + t.h - 1) / t.h;
  const int cols = cap / E / t.ntz;  // tile columns of an entry
  if (cols < 1) return false;
  t.w = std::max(kResWaves, (ux + cols - 1) / cols);
  if (kind == 0) {
    // Two blocks a CU, one computing while the other waits for its halos,
    // where that makes no more rows a CU (11 run as 12): 201x301 E=2 2.26 -> 2.05, E=8 3.7 ->
    // 3.2, E=11 5.3 -> 3.4, E=13 6.1 -> 4.7, E=16 6.2 -> 5.15; 301x921 E=2
    // 4.1 -> 3.15, E=4 7.1 -> 5.2; 90x120 E=24 3.1 -> 2.6; with a row more
    // 501x1501 E=1 3.9 -> 4.7, 301x921 E=3 5.1 -> 5.3.  In FP32, where a row
    // takes less, two tiles of 2 rows for one of 4 lose (201x301 E=5 2.83 ->
    // 2.93, 250x400 E=3 2.80 -> 2.99; exact 3.02 -> 2.83, 2.94 -> 2.76).
    const int w2 = std::max(kResWaves, (ux + 2 * cap / E / t.ntz - 1) / (2 * cap / E / t.ntz));
    const int rows = (t.w + kResWaves - 1) / kResWaves, rows2 = (w2 + kResWaves - 1) / kResWaves;
    if (2 * rows2 <= rows + (rows == 11) && (prec_ == kExact || rows2 != 2) && res_twice(rows2)) t.w = w2;
  }
  t.ntx = (ux + t.w - 1) / t.w;
  if (t.w > most) return false;
  if (resident_ == 1) return true;
  if (g_.nt < kResSteps) return false;
  if (res_rest_ > 0) return false;  // the chip is shared: a run of this handle has waited in vain
  // Measured over E (forward / backward microseconds a step, per-step kernels
  // -> resident): 201x301 E=1 4.7 -> 1.74, E=4 4.7 -> 2.7 / 8.1 -> 3.4, E=8
  // 6.2 -> 3.2 / 10.4 -> 5.2, E=11 6.9 -> 3.4 / 11.4 -> 9.1, E=16 7.9 -> 5.2,
  // E=21 9.8 -> 8.1; 301x921 E=1 5.2 -> 2.7 / 6.6 -> 3.4;
  // 501x1501 E=1 6.8 -> 4.0 / 10.4 -> 6.2.
  return true;
}

Propagator::ResLayout* Propagator::res_layout(const ResTiles& t) {
  for (auto& l : res_layouts_)
    if (l->t.w == t.w && l->t.h == t.h) return l.get();
  hipStream_t s = stream();
  auto l = std::make_unique<ResLayout>();
  l->t = t;
  const HostPoints src = bucket(src_idx_, g_.ld, t), rec = bucket(rec_idx_, g_.ld, t);
  l->fits = src.most <= kResMaxPts && rec.most <= kResMaxPts;
  const bool ok = had([&] {
    l->sptr.upload(src.ptr, s);
    l->sitems.upload(src.items, s);
    l->rptr.upload(rec.ptr, s);
    l->ritems.upload(rec.items, s);
  });
  SWFWI_HIP(hipStreamSynchronize(s));  // the host vectors end here
  if (!ok) return nullptr;
  if (res_layouts_.size() >= 16) res_layouts_.erase(res_layouts_.begin());
  res_layouts_.push_back(std::move(l));
  return res_layouts_.back().get();
}

ResGrid Propagator::res_grid(const ResTiles& t) const {
  ResGrid g;
  g.nx = g_.nxpad;
  g.nz = g_.nzpad;
  g.ld = g_.ld;
  g.nb = g_.bx0;
  g.zdamp = damp_.zdamp;
  g.bx0 = g_.bx0;
  g.bxn = g_.bxn;
  g.bz0 = g_.bz0;
  g.bzn = g_.bzn;
  g.delta_x = damp_.dx.get();
  g.delta_z = damp_.dz.get();
  g.t = t;
  return g;
}

void Propagator::res_begin(int kind, int E, int parts, ResComm& x) {
  hipStream_t s = stream();
  if (!abort_host_) {
    abort_dev_.resize(1);
    void* flag = nullptr;
    SWFWI_HIP(hipHostMalloc(&flag, sizeof(int), hipHostMallocMapped));
    abort_host_ = static_cast<int*>(flag);
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && khz > 0)
      ticks_per_us_ = khz * 1e-3;
    *abort_host_ = 1;  // cleared below
  }
  DBuf<unsigned long long>& buf = xbuf_[kind];
  const size_t words = (size_t)(kind == 1 ? 3 : 2) * E * (size_t)g_.npts();
  if (kind == 1) {
    buf.resize(std::max(words, buf.size()));
  } else if (words > buf.size() || (unsigned long long)xbase_ + (g_.nt + 1ull) * parts > 0xffffffffull) {
    // no word of the buffer carries a stamp of this run: stamps grow, and the
    // words are cleared when the buffer is new or the stamps would wrap
    buf.resize(std::max(words, buf.size()));
    launch_fill_u32(reinterpret_cast<unsigned*>(buf.get()), 2 * (long long)buf.size(), 0u, s);
    xbase_ = 0;
  }
  if (*abort_host_) {
    launch_fill(reinterpret_cast<float*>(abort_dev_.get()), 1, 0.f, s);
    *abort_host_ = 0;
  }
  x.buf = buf.get();
  x.abort_dev = abort_dev_.get();
  void* mapped = nullptr;
  SWFWI_HIP(hipHostGetDevicePointer(&mapped, abort_host_, 0));
  x.abort_host = static_cast<int*>(mapped);
  x.limit = (long long)(res_wait_us_ * ticks_per_us_);
}

void Propagator::res_part(int kind, int E, ResComm& x) {
  if (kind == 1) {
    launch_fill_u32(reinterpret_cast<unsigned*>(x.buf), 2 * 3 * E * g_.npts(), 0xffffffffu, stream());  // empty
  } else {
    x.base = xbase_;
    xbase_ += (unsigned)g_.nt + 1;
  }
}

bool Propagator::res_end(int kind, long long steps, hipEvent_t t0) {
  hipEvent_t t1 = nullptr;
  if (timing_) {
    t1 = pooled_event();
    SWFWI_HIP(hipEventRecord(t1, stream()));
  }
  SWFWI_HIP(hipGetLastError());
  SWFWI_HIP(hipStreamSynchronize(stream()));
  const bool ok = *static_cast<volatile int*>(abort_host_) == 0;
  if (ok) {
    res_pause_[kind] = kResPause;
  } else {
    gave_up++;
    res_rest_ = res_pause_[kind];
    res_pause_[kind] = std::min(2 * res_pause_[kind], kResPauseMost);
  }
  if (timing_) {
    if (ok) {
      pending_.push_back(TimedLoop{t0, t1, kind, steps});
    } else {
      event_pool_.push_back(t0);
      event_pool_.push_back(t1);
    }
  }
  return ok;
}

bool Propagator::resident_forward(int E, const float* rv, long long rvstride, const Sources& src, float* dcal,
                                  float* band, Fields& w, int rvdiv) {
  ResTiles t;
  const int parts = plan_parts(0, E, band != nullptr, t);
  if (parts < 1) return false;
  const ResLayout* l = res_layout(t);
  if (!l || !l->fits) return false;
  hipStream_t s = stream();
  const long long np = g_.npts();
  std::lock_guard<std::mutex> lock(device_lock(dev_));
  ResFwdArgs a;
  const int part = (E + parts - 1) / parts;
  if (!had([&] { res_begin(0, part, parts, a.x); })) return false;
  hipEvent_t t0 = nullptr;
  if (timing_) {
    t0 = pooled_event();
    SWFWI_HIP(hipEventRecord(t0, s));
  }
  launch_fill(w.a.get(), (long long)E * np, 0.f, s);
  launch_fill(w.b.get(), (long long)E * np, 0.f, s);
  Inject inj;
  inj.pts = src_[0].view();
  inj.amp = src.amp;
  inj.ld = src.ld;
  inj.estride = src.estride;
  inj.lo = src.lo;
  inj.hi = src.hi;
  inj.t = 0;
  launch_point_inject(w.b.get(), np, inj, g_.ns(), E, s);
  a.g = res_grid(t);
  a.nt = g_.nt;
  a.fstride = np;
  a.fa = w.a.get();
  a.fb = w.b.get();
  a.rv = rv;
  a.rvstride = rvstride;
  a.rvdiv = rvdiv;
  a.src = l->src();
  a.rec = l->rec();
  a.amp = src.amp;
  a.amp_ld = src.ld;
  a.amp_estride = src.estride;
  a.lo = src.lo;
  a.hi = src.hi;
  a.dcal = dcal;
  a.ng = g_.ng();
  a.band = band;
  a.bsize = g_.bsize;
  for (int e = 0; e < E; e += part) {
    a.g.e0 = e;
    a.E = std::min(part, E - e);
    res_part(0, a.E, a.x);
    launch_resident_fwd(a, prec_, s);
  }
  if (!res_end(0, g_.nt, t0)) return false;
  last_run[0] = LastRun{kResident, (E + part - 1) / part, t.w};
  return true;
}

bool Propagator::resident_backward(int E, const float* rv, long long rvstride, const Sources& src, const float* vsrc,
                                   long long vstride, const float* band, float* grad, long long gstride, Fields& w,
                                   int rvdiv, int it_min, const std::vector<float>& wts) {
  ResTiles t;
  const int parts = plan_parts(1, E, true, t);
  if (parts < 1) return false;
  const ResLayout* l = res_layout(t);
  if (!l || !l->fits) return false;
  hipStream_t s = stream();
  const long long np = g_.npts();
  const int nt = g_.nt, ng = g_.ng();
  if (res_wts_.size() != wts.size()) {  // the taper weights follow from dt and nt alone
    if (!had([&] { res_wts_.upload(wts, s); })) return false;
    SWFWI_HIP(hipStreamSynchronize(s));
  }
  std::lock_guard<std::mutex> lock(device_lock(dev_));
  ResBwdArgs a;
  const int part = (E + parts - 1) / parts;
  if (!had([&] { res_begin(1, part, parts, a.x); })) return false;
  hipEvent_t t0 = nullptr;
  if (timing_) {
    t0 = pooled_event();
    SWFWI_HIP(hipEventRecord(t0, s));
  }
  launch_fill(grad, (long long)E * np, 0.f, s);
  launch_fill(w.spare0, (long long)E * np, 0.f, s);
  Inject ginj;
  ginj.pts = rec_[0].view();
  ginj.amp = vsrc;
  ginj.ld = ng;
  ginj.estride = vstride;
  ginj.t = nt - 1;
  launch_point_inject(w.spare0, np, ginj, ng, E, s);
  a.g = res_grid(t);
  a.nt = nt;
  a.it_min = it_min;
  a.fstride = np;
  a.s_cur = w.s_cur;
  a.s_nxt = w.s_nxt;
  a.g_cur = w.spare0;
  a.rv = rv;
  a.rvstride = rvstride;
  a.rvdiv = rvdiv;
  a.src = l->src();
  a.rec = l->rec();
  a.amp = src.amp;
  a.amp_ld = src.ld;
  a.amp_estride = src.estride;
  a.lo = src.lo;
  a.hi = src.hi;
  a.vsrc = vsrc;
  a.ng = ng;
  a.vstride = vstride;
  a.band = band;
  a.bsize = g_.bsize;
  a.weights = res_wts_.get();
  a.grad = grad;
  a.gstride = gstride;
  for (int e = 0; e < E; e += part) {
    a.g.e0 = e;
    a.E = std::min(part, E - e);
    res_part(1, a.E, a.x);
    launch_resident_bwd(a, prec_, s);
  }
  if (!res_end(1, nt - it_min, t0)) return false;
  last_run[1] = LastRun{kResident, (E + part - 1) / part, t.w};
  return true;
}

}  // namespace swfwi

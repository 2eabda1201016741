// Step kernel of the mixed-size batch (batch.h): one launch advances every
// active entry by one time step; each wave walks one strip of one entry.
//
// A strip is up to 128 z wide (two consecutive z per lane, 116 of them outputs
// of the 10th-order step, 124 of the 4th-order one) and the wave walks it
// along x, row by row, with nothing shared with other waves and no barrier.
// The rows around the current one sit in registers (a ring of 16, the loop
// unrolled 16 times so that every ring index is a constant), so the
// x-direction terms need no memory at all; a row's z neighbours are read back
// from a row buffer in LDS that only the wave itself writes; rows of cur, prev
// and the model are loaded 4 to 5 rows ahead of their use.  The Laplacian u2
// of the row before, this one and the next follow each other in a ring of
// four, and the update lags the Laplacian by one row.
//
// What bounds it: memory in large batches (112 entries of three grid sizes,
// 29.8 M points: 72 us a step, against 101 us of the tiled form (batch_tile.hip),
// which issues about 116 vector instructions per point for staging, ring
// recomputation and index arithmetic around the ~32 of the step itself and is
// bound by them at any size); in small ones the walk itself (a lone wave issues
// one instruction per 4 cycles, about 0.35 us a row), hence the short chunks.
//
// Arithmetic (the same operations in the same order for every chunk length):
// the damped leapfrog update of fd4t10s-damp-zjh.c:14-115 in FP32 with fused
// multiply-adds, or the 4th-order leapfrog of coarse grids.
//
// Forward (FWD): the next step's source amplitude is added to `next`
// (addSource before stepForward, damp4t10d.cpp:272-289), receivers are
// recorded from cur (recordSeis after the swap), cur is stored as a snapshot
// on steps 4k+3 with the max-abs scale that the previous launch accumulated,
// and on steps before a snapshot max |next| is folded into its scale.
//
// Backward: the receiver field of calgradient (fwiframework.cpp:155-176):
// the next iteration's adjoint source is added to `next` at the receivers,
// and on iterations 4k+4 the imaging condition g -= 4 w(it) s r is formed
// with the source field C[it-1] read back from snapshot k.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "batch.h"
#include "kernels.h"
#include "march.h"

namespace swfwi {
using namespace march;
namespace {

constexpr float kF16Scale = 16384.f;  // snapshot max maps to 2^14 in FP16

// Zhang Jinhai coefficients as the reference stores them (fd4t10s-damp-zjh.c:24-29)
constexpr float kA0 = 1.53400796f, kA1 = 1.78858721f, kA2 = -0.31660756f, kA3 = 0.07612173f, kA4 = -0.01626042f,
                kA5 = 0.00216736f;

__device__ __forceinline__ unsigned short to_bf16(float x) {  // round to nearest even
  unsigned u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float from_bf16(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// Checkpoints.  Bytes a value takes, the factor it is stored with, the stores
// and loads of a lane's value, and the value read back.
template <int PREC>
constexpr unsigned kSnapBytes = PREC == kSnapF32 || PREC == kSnapNone ? 4 : 2;
template <int PREC>
__device__ __forceinline__ float snap_in(float scale) {
  if constexpr (PREC == kSnapBF16) return scale > 0.f ? 1.f / scale : 0.f;
  if constexpr (PREC == kSnapF16) return scale > 0.f ? kF16Scale / scale : 0.f;
  return 1.f;
}
template <int PREC>
__device__ __forceinline__ void snap_store(Buf b, unsigned lane_bytes, unsigned row_bytes, float v, float inv) {
  if constexpr (PREC == kSnapBF16)
    __builtin_amdgcn_raw_buffer_store_b16(to_bf16(v * inv), b, lane_bytes, row_bytes, 0);
  else if constexpr (PREC == kSnapF16)
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (_Float16)(v * inv)), b, lane_bytes,
                                          row_bytes, 0);
  else
    store1(b, lane_bytes, row_bytes, v);
}
template <int PREC>
__device__ __forceinline__ unsigned snap_load(Buf b, unsigned lane_bytes, unsigned row_bytes) {
  if constexpr (kSnapBytes<PREC> == 2)
    return __builtin_amdgcn_raw_buffer_load_b16(b, lane_bytes, row_bytes, 0);
  else
    return __builtin_amdgcn_raw_buffer_load_b32(b, lane_bytes, row_bytes, 0);
}
template <int PREC>
__device__ __forceinline__ float snap_value(unsigned s, float scale) {
  if constexpr (PREC == kSnapBF16) return from_bf16((unsigned short)s) * scale;
  if constexpr (PREC == kSnapF16)
    return (float)__builtin_bit_cast(_Float16, (unsigned short)s) * (scale * (1.f / kF16Scale));
  return __uint_as_float(s);
}

// u2 of a lane's two elements: own c (the pair), its row neighbours z, and
// the rows x-k (m[k-1]) and x+k (p[k-1]).
template <int ORDER, int R>
__device__ __forceinline__ f2 lap_pair(f2 c, const Zn<R>& z, const f2 (&m)[R], const f2 (&p)[R]) {
  f2 acc;
  if constexpr (ORDER == kOrder10) {
    constexpr float A[5] = {kA1, kA2, kA3, kA4, kA5};
    // z-k and z+k of the first and of the second element
    const float za[5] = {z.lo[0], z.lo[1], z.lo[2], z.lo[3], z.lo[4]};
    const float zb[5] = {c.x, z.lo[0], z.lo[1], z.lo[2], z.lo[3]};
    const float ya[5] = {c.y, z.hi[0], z.hi[1], z.hi[2], z.hi[3]};
    const float yb[5] = {z.hi[0], z.hi[1], z.hi[2], z.hi[3], z.hi[4]};
    acc.x = -4.f * kA0 * c.x;
    acc.y = -4.f * kA0 * c.y;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      acc.x = fmaf(A[k], (za[k] + ya[k]) + (m[k].x + p[k].x), acc.x);
      acc.y = fmaf(A[k], (zb[k] + yb[k]) + (m[k].y + p[k].y), acc.y);
    }
  } else {
    acc.x = -5.f * c.x;
    acc.y = -5.f * c.y;
    acc.x = fmaf(4.f / 3.f, (z.lo[0] + c.y) + (m[0].x + p[0].x), acc.x);
    acc.y = fmaf(4.f / 3.f, (c.x + z.hi[0]) + (m[0].y + p[0].y), acc.y);
    acc.x = fmaf(-1.f / 12.f, (z.lo[1] + z.hi[0]) + (m[1].x + p[1].x), acc.x);
    acc.y = fmaf(-1.f / 12.f, (z.lo[0] + z.hi[1]) + (m[1].y + p[1].y), acc.y);
  }
  return acc;
}

// The walk of one wave.  IMG: a backward iteration with the imaging condition.
// TAP: a forward step whose field is also kept on the 2x-coarser grid.  It is
// a kernel of its own so that the other steps carry none of it, and in the
// walk because a launch for it took 2 to 3 us: with a tap at every second step
// 12 shots of 128x64 took 1.28 ms for 200 steps so, and 1.09 ms like this.
template <int PREC, bool FWD, int ORDER, bool IMG, bool TAP>
__device__ __forceinline__ void walk(const BatchKernelArgs& a, const BatchEntry& E, int unit, int it,
                                     float (*rows)[kRowLen]) {
  constexpr int R = ORDER == kOrder10 ? 5 : 2;    // reach of u2
  constexpr int LAG = ORDER == kOrder10 ? 1 : 0;  // rows the update lags u2 by
  constexpr int HZ = R + LAG;                     // halo (even)
  constexpr int AM = kAhead - 1;
  static_assert(HZ % 2 == 0, "outputs start at a lane's first element");
  const int lane = threadIdx.x & 63;
  const int chunk = unit / E.nstrip, strip = unit - chunk * E.nstrip;
  const int xa = kHalo + chunk * E.rows, xb = min(xa + E.rows, E.nxpad - kHalo);
  const int za = kHalo + strip * E.h, zb = min(za + E.h, E.nzpad - kHalo);  // outputs [za, zb)
  const int ld = E.nzpad;
  const long long npts = (long long)E.nxpad * ld;
  const bool even = (a.rot & 1) == 0;
  const Buf cur = buffer_of((even ? a.fb : a.fa) + E.f, 4 * npts);
  const Buf nxt = buffer_of((even ? a.fa : a.fb) + E.f, 4 * npts);  // holds prev; next is written over it
  const Buf rv = buffer_of(a.rv + E.model, 4 * npts);
  // this lane's elements: z and z + 1 (lanes past the row read what follows
  // it, and past the array 0; no output depends on them)
  const int z = za - HZ + 2 * lane;
  const unsigned zo = 4u * z;
  const bool in0 = z >= za && z < zb, in1 = z + 1 >= za && z + 1 < zb;
  const bool both = in0 && in1;
  const bool odd = ((zb - za) & 1) != 0;  // the strip's last output is a lane's first element

  // sponge (fd4t10s-damp-zjh.c:64-80): by z below, by x beside; the lane's z
  // profile and, lane i, the x profile of row xa + i
  const auto profile = [&](int dist) {
    const float d = (float)dist / E.damp;
    return E.dscale * (0.05f * d * d);
  };
  const int zs = E.nzpad - E.damp;
  const bool bot0 = z >= zs, bot1 = z + 1 >= zs;
  const float dz0 = bot0 ? profile(z - zs + 1) : 0.f, dz1 = bot1 ? profile(z + 1 - zs + 1) : 0.f;
  const bool bottom = zb > zs;
  float dxl = 0.f;
  {
    const int x = xa + lane;
    if (x < E.damp) dxl = profile(E.damp - x);
    if (x >= E.nxpad - E.damp) dxl = profile(x - (E.nxpad - E.damp) + 1);
  }

  // receivers: one z, x from rx0 on.  Backward: lane i holds the amplitude of row xa + i.
  const int rx0 = E.rec0 / ld, rz = E.rec0 - rx0 * ld;
  const bool inject_next = FWD ? it + 1 < E.nt : it - 1 >= E.it_last;
  const bool rec_on = rz >= za && rz < zb && (FWD ? a.dcal != nullptr : inject_next);
  const unsigned nrec = rec_on ? E.ng : 0;  // rows rx0 .. of this strip with a receiver
  float ramp = 0.f;
  if (!FWD && rec_on) {
    const int r = xa + lane - rx0;
    if (r >= 0 && r < E.ng) ramp = a.dcal[E.dcal + (long long)(it - 1) * E.ng + r];
  }
  int sx = E.src / ld;
  const int sz = E.src - sx * ld;
  float samp = 0.f;
  if (FWD && inject_next) samp = a.amp[E.amp0 + it + 1];
  if (!FWD || !inject_next || sz < za || sz >= zb) sx = -1;

  constexpr unsigned SB = kSnapBytes<PREC>;
  const bool snap_now = FWD && PREC != kSnapNone && (it % kSnapEvery == kSnapEvery - 1);
  const bool max_now = FWD && ((it + 1) % kSnapEvery == kSnapEvery - 1) && (it + 1) / kSnapEvery < E.nsnap;
  const long long snap_off = E.snap + (long long)(FWD ? it / kSnapEvery : it / kSnapEvery - 1) * npts;
  const Buf snap = buffer_of(static_cast<char*>(a.snap) + snap_off * SB, (snap_now || IMG) ? SB * npts : 0);
  const Buf grad = buffer_of(a.grad + E.grad, 4 * npts);
  float sscale = 0.f, wimg = 0.f;
  if (snap_now) sscale = snap_in<PREC>(__uint_as_float(a.scale[E.scale0 + it / kSnapEvery]));
  if (IMG) {
    sscale = __uint_as_float(a.scale[E.scale0 + it / kSnapEvery - 1]);
    wimg = a.wts[E.wts0 + it];
  }
  // rows [plain, plain + nplain) have no sponge
  const unsigned plain = E.damp, nplain = bottom ? 0 : max(E.nxpad - 2 * E.damp, 0);
  // the coarse point of this lane: of its two elements the one in an even
  // place from row tap_oz on
  const int zt = z + ((z - E.tap_oz) & 1), kt = (zt + kHalo - E.tap_oz) >> 1;
  const bool tap_on = TAP && (zt == z ? in0 : in1) && kt < E.tap_nz;
  float* const tap = TAP ? a.tap + E.tap + (long long)a.tap_k * E.tap_nx * E.tap_nz + kt : nullptr;
  float vmax = 0.f;

  // Row of iteration i: u2 at row xa - LAG + i, update at row xa - 2 LAG + i
  // (from iteration 2 LAG on).  Ring slots: cur row y at (y - (xa - LAG - R))
  // mod 16, prev and model row y at (y - (xa - 2 LAG)) mod kAhead.
  f2 w[kRing], pv[kAhead], rm[kAhead], u[4];
  unsigned s0[kAhead], s1[kAhead];
  f2 gr[kAhead];
  const int n = xb - xa + 2 * LAG;  // iterations
  const unsigned ld4 = 4u * ld;
  const unsigned clast = (xb - 1 + HZ) * ld4, plast = (xb - 1) * ld4;  // last rows needed
  unsigned co = (xa - LAG - R) * ld4;  // next row of cur to load
  auto load_cur = [&](f2& to) {
    to = load2(cur, zo, co);
    co = min(co + ld4, clast);
  };
  unsigned po = (xa - 2 * LAG) * ld4;  // next row of prev, model, checkpoint and gradient
  auto load_own = [&](int slot) {
    pv[slot] = load2(nxt, zo, po);
    rm[slot] = load2(rv, zo, po);
    if (IMG) {
      s0[slot] = snap_load<PREC>(snap, zo / 4 * SB, po / 4 * SB);
      s1[slot] = snap_load<PREC>(snap, zo / 4 * SB + SB, po / 4 * SB);
      gr[slot] = load2(grad, zo, po);
    }
    po = min(po + ld4, plast);
  };
#pragma unroll
  for (int k = 0; k < kRing - 1; k++) load_cur(w[k]);
#pragma unroll
  for (int k = 0; k < kAhead; k++) load_own(k);

  // the z neighbours of the row of iteration i, one iteration ahead
  auto stage = [&](int buf, f2 c) {
    *reinterpret_cast<f2*>(&rows[buf][kRowPad + 2 * lane]) = c;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own rows, in order
    Zn<R> nb = z_neighbours<R>(rows[buf], lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return nb;
  };
  Zn<R> zn = stage(0, w[R]);
  unsigned yo = (xa - 2 * LAG) * ld4;  // byte offset of the updated row
  int y = xa - 2 * LAG;

  // iteration i, its place j in the ring a constant
  auto step = [&](auto place, int i) {
    constexpr int j = decltype(place)::value;
    const Zn<R> zi = zn;
    zn = stage((j + 1) & 1, w[(j + R + 1) & 15]);
    f2 m[R], p[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
      m[k] = w[(j + R - 1 - k) & 15];
      p[k] = w[(j + R + 1 + k) & 15];
    }
    u[j & 3] = lap_pair<ORDER, R>(w[(j + R) & 15], zi, m, p);
    const f2 c = w[(j + R - LAG) & 15];  // cur at the updated row
    load_cur(w[(j + 15) & 15]);
    const f2 pr = pv[j & AM], r = rm[j & AM];
    const unsigned sa = s0[j & AM], sb = s1[j & AM];
    const f2 g0 = gr[j & AM];
    load_own(j & AM);
    if (i >= 2 * LAG) {
      const f2 uc = u[(j - LAG) & 3];
      f2 v;
      if ((unsigned)y - plain >= nplain) {  // sponge
        const float dx = lane_value(dxl, y - xa);
        const float d0 = bot0 ? dz0 : dx, d1 = bot1 ? dz1 : dx;
        v.x = fmaf(2.f - 2.f * d0 + d0 * d0, c.x, -(1.f - 2.f * d0) * pr.x);
        v.y = fmaf(2.f - 2.f * d1 + d1 * d1, c.y, -(1.f - 2.f * d1) * pr.y);
      } else {
        v.x = fmaf(2.f, c.x, -pr.x);  // d = 0: the coefficients are exactly 2 and 1
        v.y = fmaf(2.f, c.y, -pr.y);
      }
      v.x = fmaf(r.x, uc.x, v.x);
      v.y = fmaf(r.y, uc.y, v.y);
      if constexpr (ORDER == kOrder10) {  // the 4th-order-in-time term r^2/12 Lap5(u2)
        const f2 um = u[(j - 2) & 3], up = u[j & 3];
        const float zm = below(uc.y), zp = above(uc.x);
        const float la = (zm + uc.y) + (um.x + up.x) - 4.f * uc.x;
        const float lb = (uc.x + zp) + (um.y + up.y) - 4.f * uc.y;
        v.x = fmaf(r.x * r.x * (1.f / 12.f), la, v.x);
        v.y = fmaf(r.y * r.y * (1.f / 12.f), lb, v.y);
      }
      const unsigned rr = (unsigned)(y - rx0);
      if constexpr (FWD) {
        if (y == sx) {
          if (z == sz) v.x += samp;
          if (z + 1 == sz) v.y += samp;
        }
        if (max_now) {
          vmax = fmaxf(vmax, in0 ? fabsf(v.x) : 0.f);
          vmax = fmaxf(vmax, in1 ? fabsf(v.y) : 0.f);
        }
        if (rr < nrec) {
          float* out = a.dcal + E.dcal + (long long)it * E.ng + rr;
          if (z == rz) *out = c.x;
          if (z + 1 == rz) *out = c.y;
        }
        if constexpr (TAP) {
          const int kx = (y + kHalo) >> 1;
          if ((y & 1) == 0 && kx < E.tap_nx && tap_on) tap[(long long)kx * E.tap_nz] = zt == z ? c.x : c.y;
        }
        if constexpr (PREC != kSnapNone) {
          if (snap_now) {
            if (in0) snap_store<PREC>(snap, zo / 4 * SB, yo / 4 * SB, c.x, sscale);
            if (in1) snap_store<PREC>(snap, zo / 4 * SB + SB, yo / 4 * SB, c.y, sscale);
          }
        }
      } else {
        if (rr < nrec) {
          const float am = lane_value(ramp, y - xa);
          if (z == rz) v.x += am;
          if (z + 1 == rz) v.y += am;
        }
        if constexpr (IMG) {
          f2 g;
          g.x = g0.x - wimg * snap_value<PREC>(sa, sscale) * c.x;
          g.y = g0.y - wimg * snap_value<PREC>(sb, sscale) * c.y;
          if (both) store2(grad, zo, yo, g);
          if (odd && in0 && !in1) store1(grad, zo, yo, g.x);
        }
      }
      if (both) store2(nxt, zo, yo, v);
      if (odd) {  // uniform
        if (in0 && !in1) store1(nxt, zo, yo, v.x);
      }
    }
    y++;
    yo += ld4;
  };
  for (int i = 0; i < n; i += kRing) {
#define SWFWI_STEP(J) \
  if (i + J >= n) break; \
  step(std::integral_constant<int, J>{}, i + J);
    SWFWI_STEP(0) SWFWI_STEP(1) SWFWI_STEP(2) SWFWI_STEP(3) SWFWI_STEP(4) SWFWI_STEP(5) SWFWI_STEP(6) SWFWI_STEP(7)
    SWFWI_STEP(8) SWFWI_STEP(9) SWFWI_STEP(10) SWFWI_STEP(11) SWFWI_STEP(12) SWFWI_STEP(13) SWFWI_STEP(14) SWFWI_STEP(15)
#undef SWFWI_STEP
  }
  if (max_now) {  // the next step's field is snapshot (it+1)/4: fold its max
    vmax = wave_max(vmax);
    // non-negative floats order like their bit patterns
    if (lane == 0) atomicMax(&a.scale[E.scale0 + (it + 1) / kSnapEvery], __float_as_uint(vmax));
  }
}

template <int PREC, bool FWD, int ORDER, bool TAP>
__global__ __launch_bounds__(64 * kWaves) void k_batch_march(BatchKernelArgs a) {
  __shared__ __align__(16) float rows[kWaves][2][kRowLen];
  // XCD-contiguous runs of the work list: blocks are dealt round-robin to the
  // 8 XCDs, so neighbouring strips and a model's shots share an XCD's L2
  const int n = a.nblocks, per = n / 8, rem = n % 8;
  const int xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = (xcd * per + (xcd < rem ? xcd : rem) + local) * kWaves + wave;
  if (l >= a.nunits) return;
  const int pk = a.blk[l];
  const BatchEntry E = a.ent[pk >> kBlkTileBits];
  const int unit = pk & ((1 << kBlkTileBits) - 1);
  const int it = FWD ? a.it_or_k : E.nt - 1 - a.it_or_k;
  if constexpr (!FWD && PREC != kSnapNone) {
    if (it >= kSnapEvery && it % kSnapEvery == 0 && a.wts[E.wts0 + it] != 0.f) {
      walk<PREC, FWD, ORDER, true, false>(a, E, unit, it, rows[wave]);
      return;
    }
  }
  walk<PREC, FWD, ORDER, false, TAP>(a, E, unit, it, rows[wave]);
}

template <bool FWD, int ORDER, bool TAP>
void launch_prec(const BatchKernelArgs& a, int prec, hipStream_t s) {
  if (a.nblocks <= 0) return;
  const dim3 grid(a.nblocks), block(64 * kWaves);
  switch (prec) {
    case kSnapF32: hipLaunchKernelGGL((k_batch_march<kSnapF32, FWD, ORDER, TAP>), grid, block, 0, s, a); break;
    case kSnapBF16: hipLaunchKernelGGL((k_batch_march<kSnapBF16, FWD, ORDER, TAP>), grid, block, 0, s, a); break;
    case kSnapF16: hipLaunchKernelGGL((k_batch_march<kSnapF16, FWD, ORDER, TAP>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_batch_march<kSnapNone, FWD, ORDER, TAP>), grid, block, 0, s, a); break;
  }
}

}  // namespace

void launch_batch_step(const BatchKernelArgs& a0, bool fwd, int prec, int order, int units, hipStream_t s) {
  BatchKernelArgs a = a0;
  a.nunits = units;
  a.nblocks = (units + kWaves - 1) / kWaves;
  const bool o4 = order == kOrder4;
  if (fwd && a.tap_k >= 0)
    o4 ? launch_prec<true, kOrder4, true>(a, prec, s) : launch_prec<true, kOrder10, true>(a, prec, s);
  else if (fwd)
    o4 ? launch_prec<true, kOrder4, false>(a, prec, s) : launch_prec<true, kOrder10, false>(a, prec, s);
  else
    o4 ? launch_prec<false, kOrder4, false>(a, prec, s) : launch_prec<false, kOrder10, false>(a, prec, s);
}

}  // namespace swfwi

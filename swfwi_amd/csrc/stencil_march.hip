// The forward step of large batches, every entry advanced by one launch, as
// strip walks (march.h): the same folded-in bookkeeping as the tiled kernel of
// stencil.hip (receivers recorded from cur, the boundary band of cur saved, the
// next step's source amplitudes added to next) and the same arithmetic bit for
// bit, with about two thirds of its vector instructions per point: nothing is
// staged or formed twice, and addresses cost nothing.
//
// What bounds it: vector issue in exact mode (about 100 instructions per two
// points, 48 of them FP64 or conversions at 4 cycles each): 60 entries of
// 301x921 with one model take 46 us a step over 400 steps and 50 over 4000, 56
// tiled over 400 (their fields alone would move in 38); 60 members of 201x301
// with a model each 17.1, 20.8 tiled.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "march.h"
#include "step_math.h"

namespace swfwi {
using namespace march;
namespace {

constexpr int R = 5;   // reach of u2
constexpr int HZ = 6;  // reach of a step
constexpr int AM = kAhead - 1;

// u2 of a lane's two elements, each ring summed as the reference does
// (((z-k + z+k) + x-k) + x+k).
template <int P>
__device__ __forceinline__ f2 u2_pair(f2 c, const Zn<R>& z, const f2 (&m)[R], const f2 (&p)[R]) {
  const float za[R] = {z.lo[0], z.lo[1], z.lo[2], z.lo[3], z.lo[4]};
  const float zb[R] = {c.x, z.lo[0], z.lo[1], z.lo[2], z.lo[3]};
  const float ya[R] = {c.y, z.hi[0], z.hi[1], z.hi[2], z.hi[3]};
  const float yb[R] = {z.hi[0], z.hi[1], z.hi[2], z.hi[3], z.hi[4]};
  float ra[R], rb[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    ra[k] = ((za[k] + ya[k]) + m[k].x) + p[k].x;
    rb[k] = ((zb[k] + yb[k]) + m[k].y) + p[k].y;
  }
  f2 u;
  u.x = u2_sum<P>(c.x, ra[0], ra[1], ra[2], ra[3], ra[4]);
  u.y = u2_sum<P>(c.y, rb[0], rb[1], rb[2], rb[3], rb[4]);
  return u;
}

// A unit's points, one per lane: its row, z and id (row -1: none, or not active
// for the entry).
struct LanePoints {
  int row, z, id, n;
};
__device__ __forceinline__ LanePoints lane_points(const UnitPoints& up, int unit, const int* lo, const int* hi, int e) {
  LanePoints p;
  const int lane = threadIdx.x & 63, b = up.ptr[unit];
  p.n = up.ptr[unit + 1] - b;
  const int first = lo ? lo[e] : 0, past = hi ? hi[e] : 0x7fffffff;
  const int4 it = lane < p.n ? up.items[b + lane] : make_int4(-1, 0, -1, 0);
  p.id = max(it.z, 0);
  p.row = it.z >= first && it.z < past ? it.x : -1;
  p.z = it.y;
  return p;
}

template <int P>
__device__ __forceinline__ void walk(const FwdStepArgs& a, const MarchMap& mm, int unit, int e, float (*rows)[kRowLen]) {
  const Grid& g = a.g;
  const int lane = threadIdx.x & 63;
  const int chunk = unit / mm.nstrip, strip = unit - chunk * mm.nstrip;
  const int xa = kHalo + chunk * mm.rows, xb = min(xa + mm.rows, g.nx - kHalo);
  const int za = kHalo + strip * mm.h, zb = min(za + mm.h, g.nz - kHalo);  // outputs [za, zb)
  const int ld = g.ld;
  const long long bytes = 4LL * g.nx * ld;
  const Buf cur = buffer_of(a.cur + (long long)e * a.fstride, bytes);
  const Buf nxt = buffer_of(a.prev + (long long)e * a.fstride, bytes);  // holds prev; next is written over it
  const Buf rv = buffer_of(a.rv + (long long)(e / a.rvdiv) * a.rvstride, bytes);
  const int z = za - HZ + 2 * lane;  // this lane's elements: z and z + 1
  const unsigned zo = 4u * z;
  const bool in0 = z >= za && z < zb, in1 = z + 1 >= za && z + 1 < zb;
  const bool both = in0 && in1;
  const bool odd = ((zb - za) & 1) != 0;  // the strip's last output is a lane's first element

  // sponge: the lane's z deltas and, lane i, the x delta of row xa + i
  const bool bot0 = z >= g.zdamp, bot1 = z + 1 >= g.zdamp;
  const float dz0 = bot0 && z < g.nz ? g.delta_z[z] : 0.f, dz1 = bot1 && z + 1 < g.nz ? g.delta_z[z + 1] : 0.f;
  const float dxl = g.delta_x[min(xa + lane, g.nx - 1)];
  const unsigned plain = g.nb, nplain = zb > g.zdamp ? 0 : max(g.nx - 2 * g.nb, 0);  // rows without sponge

  LanePoints src{-1, 0, 0, 0}, rec{-1, 0, 0, 0};
  float samp = 0.f;
  if (a.inj.t >= 0) {
    src = lane_points(mm.src, unit, a.inj.lo, a.inj.hi, e);
    if (src.n > 0 && src.row >= 0) samp = a.inj.amp[e * a.inj.estride + (long long)a.inj.t * a.inj.ld + src.id];
  }
  float* out = nullptr;
  if (a.rec.out) {
    rec = lane_points(mm.rec, unit, nullptr, nullptr, e);
    out = a.rec.out + (long long)e * a.rec.estride + rec.id;
  }
  const int rl = rec.z - (za - HZ) + kRowPad;  // the receiver's place in the row buffer

  // the boundary band (writeBndry, damp4t10d.cpp:478-514): 6 rows of x on
  // either side, 6 z at the bottom
  const int w = 6, xl = g.bx0 - w, nxb = g.nx - (xl + g.bxn - w), nzb = g.nz - g.bz0 - g.bzn, zbot = g.nz - g.bzn;
  float* band = a.band ? a.band + (long long)e * a.band_estride : nullptr;
  const unsigned nbot = band && zb > zbot ? nxb : 0;  // rows of the strip with bottom band points

  f2 wd[kRing], pv[kAhead], rm[kAhead], u[4];
  const int n = xb - xa + 2;  // iterations: u2 of row xa - 1 + i, update of row xa - 2 + i
  const unsigned ld4 = 4u * ld;
  const unsigned clast = (xb - 1 + HZ) * ld4, plast = (xb - 1) * ld4;  // last rows needed
  unsigned co = (xa - HZ) * ld4, po = (xa - 2) * ld4, yo = po;
  auto load_cur = [&](f2& to) {
    to = load2(cur, zo, co);
    co = min(co + ld4, clast);
  };
  auto load_own = [&](int slot) {
    pv[slot] = load2(nxt, zo, po);
    rm[slot] = load2(rv, zo, po);
    po = min(po + ld4, plast);
  };
#pragma unroll
  for (int k = 0; k < kRing - 1; k++) load_cur(wd[k]);
#pragma unroll
  for (int k = 0; k < kAhead; k++) load_own(k);

  // a row into the wave's buffer: its receivers are recorded from there, and
  // its z neighbours come back, one iteration ahead
  auto stage = [&](int buf, f2 c, int y) {
    *reinterpret_cast<f2*>(&rows[buf][kRowPad + 2 * lane]) = c;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own rows, in order
    Zn<R> nb = z_neighbours<R>(rows[buf], lane);
    if (rec.n > 0 && rec.row == y) *out = rows[buf][rl];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return nb;
  };
  int y = xa - 2;  // the updated row
  Zn<R> zn = stage(0, wd[R], y + 1);

  auto step = [&](auto place, int i) {
    constexpr int j = decltype(place)::value;
    const Zn<R> zi = zn;
    zn = stage((j + 1) & 1, wd[(j + R + 1) & 15], y + 2);
    f2 m[R], p[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
      m[k] = wd[(j + R - 1 - k) & 15];
      p[k] = wd[(j + R + 1 + k) & 15];
    }
    u[j & 3] = u2_pair<P>(wd[(j + R) & 15], zi, m, p);
    const f2 c = wd[(j + R - 1) & 15];  // cur at the updated row
    load_cur(wd[(j + 15) & 15]);
    const f2 pr = pv[j & AM], r = rm[j & AM];
    load_own(j & AM);
    if (i >= 2) {
      const f2 uc = u[(j - 1) & 3], um = u[(j - 2) & 3], up = u[j & 3];
      const float zm = below(uc.y), zp = above(uc.x);
      f2 v;
      if ((unsigned)y - plain >= nplain) {  // sponge
        const float dx = lane_value(dxl, y - xa);
        v.x = update_coeffs<true, P>(c.x, pr.x, r.x, cc_of(r.x), uc.x, zm, uc.y, um.x, up.x,
                                     damp_coeffs<P>(bot0 ? dz0 : dx));
        v.y = update_coeffs<true, P>(c.y, pr.y, r.y, cc_of(r.y), uc.y, uc.x, zp, um.y, up.y,
                                     damp_coeffs<P>(bot1 ? dz1 : dx));
      } else {
        const Damp<P> none{};
        v.x = update_coeffs<false, P>(c.x, pr.x, r.x, cc_of(r.x), uc.x, zm, uc.y, um.x, up.x, none);
        v.y = update_coeffs<false, P>(c.y, pr.y, r.y, cc_of(r.y), uc.y, uc.x, zp, um.y, up.y, none);
      }
      if (src.n > 0) {  // in id order (manipSource, damp4t10d.cpp:204-214)
        unsigned long long here = __ballot(src.row == y);
        while (here) {
          const int q = __builtin_ctzll(here);
          here &= here - 1;
          const float am = lane_value(samp, q);
          const int sz = __builtin_amdgcn_readlane(src.z, q);
          if (z == sz) v.x = a.inj.sign > 0 ? v.x + am : v.x - am;
          if (z + 1 == sz) v.y = a.inj.sign > 0 ? v.y + am : v.y - am;
        }
      }
      if (band) {
        int col = -1;  // of the six on either side
        if ((unsigned)(y - xl) < (unsigned)w) col = y - xl;
        if ((unsigned)(y - (g.nx - g.bxn)) < (unsigned)w) col = y - (g.nx - g.bxn) + w;
        if (col >= 0) {
          float* to = band + w * nxb + (long long)nzb * col - g.bz0;
          if (in0 && z < zbot) to[z] = c.x;
          if (in1 && z + 1 < zbot) to[z + 1] = c.y;
        }
        if ((unsigned)(y - xl) < nbot) {
          float* to = band + (long long)w * (y - xl) - zbot;
          if (in0 && z >= zbot && z < zbot + w) to[z] = c.x;
          if (in1 && z + 1 >= zbot && z + 1 < zbot + w) to[z + 1] = c.y;
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
#define SWFWI_STEP(J)    \
  if (i + J >= n) break; \
  step(std::integral_constant<int, J>{}, i + J);
    SWFWI_STEP(0) SWFWI_STEP(1) SWFWI_STEP(2) SWFWI_STEP(3) SWFWI_STEP(4) SWFWI_STEP(5) SWFWI_STEP(6) SWFWI_STEP(7)
    SWFWI_STEP(8) SWFWI_STEP(9) SWFWI_STEP(10) SWFWI_STEP(11) SWFWI_STEP(12) SWFWI_STEP(13) SWFWI_STEP(14) SWFWI_STEP(15)
#undef SWFWI_STEP
  }
}

template <int P>
__global__ __launch_bounds__(64 * kWaves) void k_fwd_march(FwdStepArgs a, MarchMap mm, int nentries) {
  __shared__ __align__(16) float rows[kWaves][2][kRowLen];
  // XCD-contiguous runs of the work list.  Entries that share a model come
  // back to back (its rows are then read from the XCD's L2), entries with
  // models of their own one after the other (neighbouring strips and chunks
  // share rows of cur).
  const int n = gridDim.x, per = n / 8, rem = n % 8;
  const int xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = (xcd * per + (xcd < rem ? xcd : rem) + local) * kWaves + wave;
  const int units = mm.nstrip * mm.nchunk;
  if (l >= units * nentries) return;
  int unit, e;
  if (mm.shared) {
    unit = l / nentries;
    e = l - unit * nentries;
  } else {
    e = l / units;
    unit = l - e * units;
  }
  walk<P>(a, mm, unit, e, rows[wave]);
}

}  // namespace

void launch_fwd_march(const FwdStepArgs& a, const MarchMap& m, int nentries, int precision, hipStream_t s) {
  const long long waves = (long long)m.nstrip * m.nchunk * nentries;
  const dim3 grid((unsigned)((waves + kWaves - 1) / kWaves)), block(64 * kWaves);
  if (precision == kExact)
    hipLaunchKernelGGL(k_fwd_march<kExact>, grid, block, 0, s, a, m, nentries);
  else
    hipLaunchKernelGGL(k_fwd_march<kFp32>, grid, block, 0, s, a, m, nentries);
}

}  // namespace swfwi

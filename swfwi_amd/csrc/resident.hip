// Kernels of the resident time loop (resident.h).
//
// Lane l of a wave is z = z0 - 1 + l, so the u2 values a row's update needs at
// z +- 1 sit in the neighbouring lanes (whole-wave DPP shifts) and the ring
// columns z0-1 and z0+h are computed by lanes that would otherwise idle.  Wave
// w owns the tile's rows [w*R, w*R + R): their u2 stays in registers, and only
// each wave's first and last u2 row pass through LDS for the waves beside it.
// The ring rows -1 and w (the tile's width) are formed by the waves at the
// ends.  Two barriers per step: cur complete (own rows and halo) -> u2 ->
// barrier -> update, publish, collect the halo -> barrier.
//
// What bounds a step: the exchange (a store past the L2, the neighbour's poll:
// 1.4-2.3 us on its own, measured without stencil work) and, on wide tiles, the
// arithmetic (about 0.3 us per row of a wave).  Forward 1.74 / 2.7 / 4.0 us a
// step on the 201x301 / 301x921 / 501x1501 grids, against 4.7 / 5.2 / 6.8 as
// launches; backward 3.4 / 6.2 on the last two, against 6.6 / 10.4.
#include "resident.h"

#include "step_math.h"

namespace swfwi {
namespace {

typedef unsigned long long u64;
constexpr int LZ = kResLdz;

// the value of the lane below / above (z - 1 / z + 1); the end lanes get 0
__device__ __forceinline__ float lane_below(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_above(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}

// Element i of an array with a block-uniform base, the byte offset in 32 bits.
template <class T>
__device__ __forceinline__ T& elem(T* p, unsigned i) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return *reinterpret_cast<T*>(reinterpret_cast<B*>(p) + i * (unsigned)sizeof(T));
}
// Makes a loop-invariant value opaque to the compiler in each iteration, so
// that what is derived from it (a lane mask per row, a coefficient) is formed
// where it is used instead of being kept, and spilled, across the loop.
__device__ __forceinline__ void refresh(unsigned& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void refresh(float& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ void put(u64* p, float v, unsigned stamp) {
  __hip_atomic_store(p, ((u64)stamp << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 peek(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// u2 of a row: s is the lane's element of the row in LDS (z neighbours at
// +-k), w[0..10] the column at x-5..x+5.
template <int P>
__device__ __forceinline__ float u2_row(const float* __restrict__ s, const float* __restrict__ w) {
  const float r1 = ((s[-1] + s[1]) + w[4]) + w[6];
  const float r2 = ((s[-2] + s[2]) + w[3]) + w[7];
  const float r3 = ((s[-3] + s[3]) + w[2]) + w[8];
  const float r4 = ((s[-4] + s[4]) + w[1]) + w[9];
  const float r5 = ((s[-5] + s[5]) + w[0]) + w[10];
  return u2_sum<P>(w[5], r1, r2, r3, r4, r5);
}

// Where a block works: entry, tile, its extent and this thread's place in it.
// (tid: the thread among those of its field, of which there are 64 * waves).
struct Place {
  int e, tile, x0, z0, w, h, wave, lane, row0, tid;
};
template <int NW>
__device__ __forceinline__ Place place(const ResGrid& g, int rows) {
  Place p;
  const int nt = g.t.ntx * g.t.ntz;
  const int e = blockIdx.x / nt;
  p.e = g.e0 + e;
  p.tile = blockIdx.x - e * nt;
  const int tx = p.tile / g.t.ntz, tz = p.tile - tx * g.t.ntz;
  p.x0 = kHalo + tx * g.t.w;
  p.z0 = kHalo + tz * g.t.h;
  p.w = min(g.t.w, g.nx - kHalo - p.x0);
  p.h = min(g.t.h, g.nz - kHalo - p.z0);
  p.lane = threadIdx.x & 63;
  p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % NW;
  p.tid = threadIdx.x % (64 * NW);
  p.row0 = p.wave * rows;
  return p;
}

// This thread's share of the tile's halo: the 6 rows on either side, the 6
// columns above and below, and the corner points that the u2 ring reads (row
// or column 1 beyond the tile, up to 5 beyond in the other direction).  Only
// points the propagation updates; the grid's rim stays zero in LDS.
template <int NH>
struct Halo {
  unsigned q[NH];  // grid index
  int l[NH];       // LDS index
  unsigned on;     // bit j: point j exists
};
template <int NT, int NH>
__device__ __forceinline__ void halo_points(const ResGrid& g, const Place& p, Halo<NH>& hp) {
  const int nside = 12 * p.h, nend = 12 * p.w, ntot = nside + nend + 36;
  hp.on = 0;
#pragma unroll
  for (int j = 0; j < NH; j++) {
    const int i = (int)threadIdx.x + j * NT;
    int rx = 0, rz = 0;  // tile coordinates
    if (i < nside) {
      const int r = i / p.h;
      rz = i - r * p.h;
      rx = r < 6 ? r - 6 : p.w + r - 6;
    } else if (i < nside + nend) {
      const int k = i - nside, r = k % 12;
      rx = k / 12;
      rz = r < 6 ? r - 6 : p.h + r - 6;
    } else if (i < ntot) {
      const int k = i - nside - nend, c = k / 9, m = k % 9;
      const int dx = m < 5 ? 1 : m - 3, dz = m < 5 ? m + 1 : 1;  // (1, 1..5), (2..5, 1)
      rx = (c & 1) ? p.w - 1 + dx : -dx;
      rz = (c & 2) ? p.h - 1 + dz : -dz;
    }
    const int gx = p.x0 + rx, gz = p.z0 + rz;
    const bool ok = i < ntot && gx >= kHalo && gx < g.nx - kHalo && gz >= kHalo && gz < g.nz - kHalo;
    hp.q[j] = ok ? (unsigned)(gx * g.ld + gz) : 0u;
    hp.l[j] = ok ? (rx + 6) * LZ + rz + 6 : 0;
    if (ok) hp.on |= 1u << j;
  }
}

// A block's first look at its halo waits this long (x 64 cycles, about 0.3 us):
// its neighbours publish when it does and a word takes that long to get there,
// so an earlier look only adds a round trip and traffic (0 / 8 / 12 / 16 / 24:
// 1.88 / 1.78 / 1.74 / 1.78 / 1.98 us a step on the 201x301 grid, 4.48 / 3.97 /
// 3.92 / 3.98 / 4.17 on the 501x1501 one).
constexpr int kFirstPoll = 12;

// Whether a wait has to end: it ran out of time (t0: when it began, 0 at the
// first look) or another block gave up.
__device__ __forceinline__ bool give_up(const ResComm& x, int spin, long long& t0) {
  if ((spin & 63) != 63 && x.limit != 0) return false;
  const long long now = wall_clock64();
  if (t0 == 0) t0 = now;
  if (now - t0 < x.limit && __hip_atomic_load(x.abort_dev, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    return false;
  __hip_atomic_store(x.abort_dev, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(x.abort_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  return true;
}

// Collects the halo words of stamp `want` into LDS; false when the wait ran
// out or another block gave up.
template <int NH>
__device__ __forceinline__ bool collect(const ResComm& x, const u64* words, Halo<NH>& hp, unsigned want, float* c) {
  u64 v[NH];
  refresh(hp.on);
  __builtin_amdgcn_s_sleep(kFirstPoll);
  long long t0 = 0;
  for (int spin = 0;; spin++) {
    bool all = true;
#pragma unroll
    for (int j = 0; j < NH; j++) v[j] = (hp.on >> j) & 1 ? peek(&elem(words, hp.q[j])) : (u64)want << 32;
#pragma unroll
    for (int j = 0; j < NH; j++) all = all && (unsigned)(v[j] >> 32) == want;
    if (all) break;
    if (give_up(x, spin, t0)) return false;
  }
#pragma unroll
  for (int j = 0; j < NH; j++)
    if ((hp.on >> j) & 1) c[hp.l[j]] = __uint_as_float((unsigned)v[j]);
  return true;
}

// The exchange of two fields: a point's two values in one word, empty words
// all ones (a pair of that NaN would wait until the limit).  Three copies in
// turn: while step k is formed a block empties its words of the copy that step
// k + 1 will use; every reader has taken step k - 2 from it by then, and none
// looks for k + 1 before it has k, which the block publishes only when its
// emptying stores have arrived.  Two stamped words a point move twice the
// bytes: 2.8 against 2.3 us a step for the exchange alone on the 301x921 grid,
// 4.3 against 3.1 on the 501x1501 one (one field is faster stamped, 1.75
// against 2.0 us: it has no emptying to wait for).
constexpr u64 kEmpty = ~(u64)0;
__device__ __forceinline__ void put_pair(u64* p, float s, float g) {
  __hip_atomic_store(p, ((u64)__float_as_uint(g) << 32) | __float_as_uint(s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int NH>
__device__ __forceinline__ bool collect_pairs(const ResComm& x, const u64* words, Halo<NH>& hp, float* s, float* g) {
  u64 v[NH];
  refresh(hp.on);
  __builtin_amdgcn_s_sleep(kFirstPoll);
  long long t0 = 0;
  for (int spin = 0;; spin++) {
    bool all = true;
#pragma unroll
    for (int j = 0; j < NH; j++) v[j] = (hp.on >> j) & 1 ? peek(&elem(words, hp.q[j])) : 0;
#pragma unroll
    for (int j = 0; j < NH; j++) all = all && v[j] != kEmpty;
    if (all) break;
    if (give_up(x, spin, t0)) return false;
  }
#pragma unroll
  for (int j = 0; j < NH; j++)
    if ((hp.on >> j) & 1) {
      s[hp.l[j]] = __uint_as_float((unsigned)v[j]);
      g[hp.l[j]] = __uint_as_float((unsigned)(v[j] >> 32));
    }
  return true;
}

// A tile's point list in LDS: place (-1: not active for the entry), the next
// active point of the same place (kNone: none) and, for injections, two steps'
// amplitudes.
constexpr unsigned kNone = 0xffff;
struct Points {
  int loc[kResMaxPts];
  unsigned short next[kResMaxPts];
  float amp[2][kResMaxPts];
};
// n points; threads 0..n-1 hold one each (place and id)
__device__ __forceinline__ int points_begin(const ResPoints& pl, const Place& p, const int* lo, const int* hi, int& loc,
                                            int& pid) {
  const int b = pl.ptr[p.tile], n = pl.ptr[p.tile + 1] - b;
  const int first = lo ? lo[p.e] : 0, past = hi ? hi[p.e] : 0x7fffffff;
  const int2 it = p.tid < n ? pl.items[b + p.tid] : make_int2(-1, -1);
  pid = max(it.y, 0);
  loc = it.y >= first && it.y < past ? it.x : -1;
  return n;
}
// The first active point at each of the thread's rows, two 16-bit indices a
// register (kNone: no point), once the list is in LDS.
template <int R>
struct Heads {
  unsigned h[(R + 1) / 2];
  __device__ __forceinline__ void fresh() {
#pragma unroll
    for (int i = 0; i < (R + 1) / 2; i++) refresh(h[i]);
  }
  __device__ __forceinline__ unsigned at(int k) const { return (h[k >> 1] >> (16 * (k & 1))) & 0xffffu; }
};
template <int R>
__device__ __forceinline__ void find_heads(const Points& pt, int n, const Place& p, Heads<R>& hd) {
#pragma unroll
  for (int i = 0; i < (R + 1) / 2; i++) hd.h[i] = 0xffffffffu;
  for (int j = n - 1; j >= 0; j--) {
    const int loc = pt.loc[j], k = (loc >> 6) - p.row0;
    if (loc < 0 || (loc & 63) != p.lane || k < 0 || k >= R) continue;
#pragma unroll
    for (int i = 0; i < (R + 1) / 2; i++)
      if (i == k >> 1) hd.h[i] = (k & 1) ? (hd.h[i] & 0xffffu) | ((unsigned)j << 16) : (hd.h[i] & 0xffff0000u) | (unsigned)j;
  }
}
// Links thread j's point to the next active one of its place; true if there is one.
__device__ __forceinline__ bool link(Points& pt, int n, int j) {
  const int loc = pt.loc[j];
  int i = loc < 0 ? n : j + 1;
  while (i < n && pt.loc[i] != loc) i++;
  pt.next[j] = i < n ? (unsigned short)i : (unsigned short)kNone;
  return i < n;
}
// Adds (or subtracts) the amplitude of head h; where points of the tile share
// places, every one of the place in id order, along the links.  (A scan of the
// rest of the list in their place held the whole tile up: 1561 receivers on 1501
// places of the 501x1501 grid 31 us a backward iteration, 7.5 with the links, 11.4
// as launches; 480 sources on 12 places of 201x301 36 us a step, 4.6 with them.)
__device__ __forceinline__ float inject(const Points& pt, int slot, unsigned h, bool shared, bool add, float v) {
  v = add ? v + pt.amp[slot][h] : v - pt.amp[slot][h];
  if (shared)
    for (unsigned j = pt.next[h]; j != kNone; j = pt.next[j]) v = add ? v + pt.amp[slot][j] : v - pt.amp[slot][j];
  return v;
}

__device__ __forceinline__ int band_at(const ResGrid& g, int ix, int iz) {
  const int w = 6, xl = g.bx0 - w, nxb = g.nx - (g.bx0 - w + g.bxn - w), nzb = g.nz - g.bz0 - g.bzn, zb = g.nz - g.bzn;
  if (iz >= zb && iz < zb + w && ix >= xl && ix < xl + nxb) return (iz - zb) + w * (ix - xl);
  if (iz >= g.bz0 && iz < g.bz0 + nzb) {
    if (ix >= xl && ix < g.bx0) return w * nxb + (iz - g.bz0) + nzb * (ix - xl);
    const int xr = g.nx - g.bxn;
    if (ix >= xr && ix < xr + w) return w * nxb + (iz - g.bz0) + nzb * (ix - xr + w);
  }
  return -1;
}

// The sponge of a tile: coefficients by row (x sponge, in LDS) and of the
// thread's z (bottom sponge, which wins).
template <int P>
struct Sponge {
  Damp<P> z;
  bool bottom;
};
template <int P>
__device__ __forceinline__ Sponge<P> sponge_begin(const ResGrid& g, const Place& p, int iz, bool zin, Damp<P>* rows) {
  Sponge<P> s;
  s.bottom = zin && iz >= g.zdamp;
  s.z = damp_coeffs<P>(s.bottom ? g.delta_z[iz] : 0.f);
  if (p.tid < p.w) rows[p.tid] = damp_coeffs<P>(g.delta_x[p.x0 + p.tid]);
  return s;
}
template <int P>
__device__ __forceinline__ Damp<P> sponge_at(const Sponge<P>& s, const Damp<P>* rows, int row) {
  const Damp<P> x = rows[row];
  return Damp<P>{s.bottom ? s.z.a : x.a, s.bottom ? s.z.b : x.b};
}

// cur of the tile and its halo from a field in memory into LDS (zeroed before).
template <int NW>
__device__ __forceinline__ void load_tile(const ResGrid& g, const Place& p, const float* __restrict__ f, float* c) {
  for (int r = p.wave; r < p.w + 12; r += NW) {
    const float* src = f + (long long)(p.x0 - 6 + r) * g.ld + p.z0 - 6;
    for (int z = p.lane; z < p.h + 12; z += 64) c[r * LZ + z] = src[z];
  }
}

// The u2 rows of a wave: u[1 + k] of its row k, and, where the wave is at the
// tile's end, the ring row beside it (u[0], u[R + 1]).  The first and last row
// go to LDS (ub) for the waves beside.  win: the wave's column, rows row0 - 5
// .. row0 + R + 4.
template <int P, int R>
__device__ __forceinline__ void form_rows(const float* cur, const Place& p, const float (&win)[R + 10], float (&u)[R + 2],
                                          float* ub) {
  const float* c = cur + (p.row0 + 6) * LZ + p.lane + 5;
  u[0] = u[R + 1] = 0.f;
#pragma unroll
  for (int k = 0; k < R; k++) {
    // the row's offset through an empty asm, so that its z reads share one address register
    int o = k * LZ;
    asm("" : "+v"(o));
    u[k + 1] = u2_row<P>(c + o, win + k);
    // no more rows in flight than the registers hold
    if (R > 3 && (k & 1)) __builtin_amdgcn_sched_barrier(0);
  }
  if (p.wave == 0) {
    float e[11];
    e[0] = c[-6 * LZ];
#pragma unroll
    for (int i = 1; i < 11; i++) e[i] = win[i - 1];
    u[0] = u2_row<P>(c - LZ, e);
  }
  if (p.row0 + R == p.w) {  // the next row is the ring's
    float e[11];
    e[10] = c[(R + 5) * LZ];
#pragma unroll
    for (int i = 0; i < 10; i++) e[i] = win[R + i];
    u[R + 1] = u2_row<P>(c + R * LZ, e);
  }
  ub[(2 * p.wave) * 64 + p.lane] = u[1];
  ub[(2 * p.wave + 1) * 64 + p.lane] = u[R];
}
// after the barrier: the rows beside the wave's, from the waves beside
template <int NW, int R>
__device__ __forceinline__ void ring_rows(const Place& p, float (&u)[R + 2], const float* ub) {
  if (p.wave > 0) u[0] = ub[(2 * p.wave - 1) * 64 + p.lane];
  if (p.wave + 1 < NW && p.row0 + R < p.w) u[R + 1] = ub[(2 * p.wave + 2) * 64 + p.lane];
}

// the most halo points of a tile of up to w columns per thread of NT
constexpr int halo_share(int w, int NT) { return (12 * kResTileZ + 12 * w + 36 + NT - 1) / NT; }

// This thread's share of the points a tile publishes: those within 6 of its edges.
template <int NT, int NE>
__device__ __forceinline__ void edge_points(const ResGrid& g, const Place& p, Halo<NE>& ep) {
  const int rows = min(p.w, 12), cols = min(p.h, 12);  // edge rows; edge columns of the rows between
  const int nrow = rows * p.h, ntot = nrow + (p.w - rows) * cols;
  ep.on = 0;
#pragma unroll
  for (int j = 0; j < NE; j++) {
    const int i = (int)threadIdx.x + j * NT;
    int rx = 0, rz = 0;
    if (i < nrow) {
      const int r = i / p.h;
      rz = i - r * p.h;
      rx = r < 6 ? r : p.w - rows + r;
    } else if (i < ntot) {
      const int k = i - nrow, r = k % cols;
      rx = 6 + k / cols;
      rz = r < 6 ? r : p.h - cols + r;
    }
    const bool ok = i < ntot;
    ep.q[j] = ok ? (unsigned)((p.x0 + rx) * g.ld + p.z0 + rz) : 0u;
    ep.l[j] = ok ? (rx + 6) * LZ + rz + 6 : 0;
    if (ok) ep.on |= 1u << j;
  }
}
constexpr int edge_share(int w, int NT) {
  return ((w <= 12 ? w * kResTileZ : 12 * kResTileZ + (w - 12) * 12) + NT - 1) / NT;
}

// (tiles of up to kResTwiceRows rows a wave in 128 registers, so that two
// blocks fit a CU; 5 and 6 rows spill 3 and 23 of them)
template <int P, int R, int NW>
__global__ __launch_bounds__(64 * NW, R <= kResTwiceRows ? 4 : 2) void k_resident_fwd(ResFwdArgs a) {
  constexpr int NX = NW * R + 12;
  __shared__ float cur[NX * LZ];
  __shared__ float ub[2 * NW * 64];
  __shared__ Damp<P> rows[NW * R];
  __shared__ Points sp;
  __shared__ int dead, shared;
  const ResGrid& g = a.g;
  const Place p = place<NW>(g, R);
  const long long fo = (long long)p.e * a.fstride;
  if (threadIdx.x == 0) dead = shared = 0;
  for (int i = threadIdx.x; i < NX * LZ; i += 64 * NW) cur[i] = 0.f;
  int sloc, spid, rloc, rpid = 0;
  const int ns = points_begin(a.src, p, a.lo, a.hi, sloc, spid);
  const int nr = a.dcal ? points_begin(a.rec, p, nullptr, nullptr, rloc, rpid) : 0;
  const bool has_src = p.tid < ns, has_rec = p.tid < nr;
  const float* amp = a.amp + p.e * a.amp_estride;
  if (has_src) {
    sp.loc[p.tid] = sloc;
    if (a.nt > 1) sp.amp[1][p.tid] = amp[a.amp_ld + spid];
  }
  float* rec = a.dcal + (long long)p.e * a.nt * a.ng;
  const int rl = has_rec ? ((rloc >> 6) + 6) * LZ + (rloc & 63) + 5 : 0;
  // this lane's points
  const bool zin = p.lane >= 1 && p.lane <= p.h;
  const int iz = p.z0 - 1 + p.lane;
  const float* rvp = a.rv + (long long)(p.e / a.rvdiv) * a.rvstride;
  const bool sponge = p.x0 < g.nb || p.x0 + p.w > g.nx - g.nb || p.z0 + p.h > g.zdamp;
  const Sponge<P> damp = sponge_begin<P>(g, p, iz, zin, rows);
  float prv[R], rv[R];
  int bi[R];
  unsigned edge = 0, inband = 0;  // bit k: row k's point is published / in the boundary band
  unsigned q0 = (unsigned)((p.x0 + p.row0) * g.ld + iz);
  __syncthreads();
  load_tile<NW>(g, p, a.fb + fo, cur);
  if (has_src && link(sp, ns, p.tid)) shared = 1;
  Heads<R> head;
  find_heads<R>(sp, ns, p, head);
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = p.row0 + k;
    const bool in = zin && row < p.w;
    prv[k] = in ? a.fa[fo + q0 + k * g.ld] : 0.f;
    rv[k] = in ? rvp[q0 + k * g.ld] : 0.f;
    bi[k] = in && a.band ? band_at(g, p.x0 + row, iz) : -1;
    if (bi[k] >= 0) inband |= 1u << k;
    if (in && (p.lane <= 6 || p.lane > p.h - 6 || row < 6 || row >= p.w - 6)) edge |= 1u << k;
  }
  const bool band_tile = __ballot(inband != 0) != 0;  // uniform over the wave
  float* band = a.band + (long long)p.e * a.nt * a.bsize;
  constexpr int NH = halo_share(NW * R, 64 * NW);
  Halo<NH> hp;
  halo_points<64 * NW, NH>(g, p, hp);
  const long long words = (long long)a.E * a.fstride;  // of one parity
  const long long xo = (long long)(p.e - g.e0) * a.fstride;
  __syncthreads();
  const bool chains = shared != 0;

  for (int it = 0; it < a.nt; it++) {
    refresh(edge);
    refresh(q0);
    head.fresh();
    float win[R + 10], u[R + 2];
    {
      const float* c = cur + (p.row0 + 1) * LZ + p.lane + 5;
#pragma unroll
      for (int k = 0; k < R + 10; k++) win[k] = c[k * LZ];
    }
    float anext = 0.f;
    if (has_src && it + 2 < a.nt) anext = elem(amp + (long long)(it + 2) * a.amp_ld, spid);
    form_rows<P, R>(cur, p, win, u, ub);
    if (has_rec) elem(rec + (long long)it * a.ng, rpid) = cur[rl];
    if (band_tile) {
      refresh(inband);
#pragma unroll
      for (int k = 0; k < R; k++)
        if ((inband >> k) & 1) elem(band + (long long)it * a.bsize, bi[k]) = win[k + 5];
    }
    __syncthreads();
    ring_rows<NW, R>(p, u, ub);
    const unsigned stamp = a.x.base + (unsigned)it + 1;
    u64* words_now = a.x.buf + ((it + 1) & 1) * words + xo;
    const bool more = it + 1 < a.nt;
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int row = p.row0 + k;
      if (row < p.w) {  // wave-uniform
        const float c = win[k + 5], zm = lane_below(u[k + 1]), zp = lane_above(u[k + 1]);
        if (R > 4) refresh(rv[k]);
        const float cc = cc_of(rv[k]);
        float v = sponge ? update_coeffs<true, P>(c, prv[k], rv[k], cc, u[k + 1], zm, zp, u[k], u[k + 2],
                                                  sponge_at<P>(damp, rows, row))
                         : update_coeffs<false, P>(c, prv[k], rv[k], cc, u[k + 1], zm, zp, u[k], u[k + 2], damp.z);
        if (ns > 0 && more) {
          const unsigned h = head.at(k);
          if (h != kNone) v = inject(sp, (it + 1) & 1, h, chains, true, v);
        }
        prv[k] = c;
        if (zin) {
          if (more && ((edge >> k) & 1)) put(&elem(words_now, q0 + k * g.ld), v, stamp);
          cur[(row + 6) * LZ + p.lane + 5] = v;
        }
      }
    }
    if (has_src) sp.amp[it & 1][p.tid] = anext;
    if (more && !collect<NH>(a.x, words_now, hp, stamp, cur)) dead = 1;
    __syncthreads();
    if (dead) return;
  }
  // p(nt-1) in prv, p(nt) in LDS
  float* newest = ((a.nt & 1) ? a.fa : a.fb) + fo;
  float* older = ((a.nt & 1) ? a.fb : a.fa) + fo;
#pragma unroll
  for (int k = 0; k < R; k++)
    if (zin && p.row0 + k < p.w) {
      newest[q0 + k * g.ld] = cur[(p.row0 + k + 6) * LZ + p.lane + 5];
      older[q0 + k * g.ld] = prv[k];
    }
}

// The backward iteration with a field per half of the block: waves 0-7 the
// source field (undamped step, subSource, imaging condition, band restore),
// waves 8-15 the receiver field (damped step, injection); a wave with both
// fields has twice the chain and runs out of registers at 6 rows (301x921 4.8 us
// a step, 501x1501 14).  Once both new fields are in LDS all 16 waves publish
// the tile's edge as a list, a pair a thread, and collect the halo.  Both halves
// run the same barriers.  (The forward kernel publishes from its registers: the
// list there costs a barrier and gains nothing, 2.83 against 2.72 us.)
template <int P, int R>
struct BwdTile {
  static constexpr int NW = kResWaves, NX = NW * R + 12;
  float f[2][NX * LZ];
  float ub[2][2 * NW * 64];
  Damp<P> rows[NW * R];
  Points pt[2];
  int dead, shared[2];
};
template <int P, int R, bool SRC>
__device__ __forceinline__ void bwd_half(const ResBwdArgs& a, BwdTile<P, R>& t) {
  constexpr int NW = kResWaves;
  constexpr int F = SRC ? 0 : 1;
  const ResGrid& g = a.g;
  const Place p = place<NW>(g, R);
  const long long fo = (long long)p.e * a.fstride;
  float* cur = t.f[F];
  Points& pt = t.pt[F];
  if (p.tid == 0) {
    t.shared[F] = 0;
    if (SRC) t.dead = 0;
  }
  for (int i = p.tid; i < BwdTile<P, R>::NX * LZ; i += 64 * NW) cur[i] = 0.f;
  int loc, pid;
  const int n = points_begin(SRC ? a.src : a.rec, p, SRC ? a.lo : nullptr, SRC ? a.hi : nullptr, loc, pid);
  const bool has = p.tid < n;
  const int last = a.nt - 1;
  // the sources of iteration it enter in it, the receivers' of it - 1
  const float* amp = SRC ? a.amp + p.e * a.amp_estride : a.vsrc + p.e * a.vstride - a.ng;
  const int amp_ld = SRC ? a.amp_ld : a.ng;
  if (has) {
    pt.loc[p.tid] = loc;
    if (SRC || last - 1 >= a.it_min) pt.amp[last & 1][p.tid] = amp[(long long)last * amp_ld + pid];
  }
  const bool zin = p.lane >= 1 && p.lane <= p.h;
  const int iz = p.z0 - 1 + p.lane;
  const float* rvp = a.rv + (long long)(p.e / a.rvdiv) * a.rvstride;
  const bool sponge = !SRC && (p.x0 < g.nb || p.x0 + p.w > g.nx - g.nb || p.z0 + p.h > g.zdamp);
  Sponge<P> damp{};
  if (!SRC) damp = sponge_begin<P>(g, p, iz, zin, t.rows);
  __syncthreads();
  load_tile<NW>(g, p, (SRC ? a.s_cur : a.g_cur) + fo, cur);
  if (has && link(pt, n, p.tid)) t.shared[F] = 1;
  Heads<R> head;
  find_heads<R>(pt, n, p, head);
  float prv[R], rv[R], grad[R], bv[R];
  int bi[R];
  unsigned inband = 0;
  const float* band = a.band + (long long)p.e * a.nt * a.bsize;
  const unsigned q0 = (unsigned)((p.x0 + p.row0) * g.ld + iz);
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = p.row0 + k;
    const bool in = zin && row < p.w;
    prv[k] = SRC && in ? a.s_nxt[fo + q0 + k * g.ld] : 0.f;
    rv[k] = in ? rvp[q0 + k * g.ld] : 0.f;
    grad[k] = 0.f;
    bi[k] = SRC && in ? band_at(g, p.x0 + row, iz) : -1;
    if (bi[k] >= 0) inband |= 1u << k;
    bv[k] = bi[k] >= 0 && last - 1 >= a.it_min ? band[(long long)(last - 1) * a.bsize + bi[k]] : 0.f;
  }
  const bool band_tile = SRC && __ballot(inband != 0) != 0;  // uniform over the wave
  constexpr int NT = 2 * 64 * NW, NH = halo_share(NW * R, NT), NE = edge_share(NW * R, NT);
  Halo<NH> hp;
  Halo<NE> ep;
  halo_points<NT, NH>(g, p, hp);
  edge_points<NT, NE>(g, p, ep);
  const long long copy = (long long)a.E * a.fstride;  // words of one of the three copies
  u64* words = a.x.buf + (long long)(p.e - g.e0) * a.fstride;
  int turn = 0;  // the copy that the field being formed goes to
  __syncthreads();
  const bool chains = t.shared[F] != 0;

  for (int it = last; it >= a.it_min; it--) {
    const bool more = it - 1 >= a.it_min, more2 = it - 2 >= a.it_min;
    refresh(inband);
    refresh(ep.on);
    head.fresh();
    const int next = turn == 2 ? 0 : turn + 1;
    if (more2) {
#pragma unroll
      for (int j = 0; j < NE; j++)
        if ((ep.on >> j) & 1)
          __hip_atomic_store(&elem(words + next * copy, ep.q[j]), kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float win[R + 10], u[R + 2], rc[R];
    float anext = 0.f, weight = 0.f;
    if (has && (SRC ? more : more2)) anext = elem(amp + (long long)(it - 1) * amp_ld, pid);
    if (SRC) weight = a.weights[it];
    {
      const float* c = cur + (p.row0 + 1) * LZ + p.lane + 5;
#pragma unroll
      for (int k = 0; k < R + 10; k++) win[k] = c[k * LZ];
    }
    form_rows<P, R>(cur, p, win, u, t.ub[F]);
    if (SRC) {  // the receiver field at this half's points, before its half moves on
#pragma unroll
      for (int k = 0; k < R; k++) rc[k] = t.f[1][(p.row0 + k + 6) * LZ + p.lane + 5];
    }
    __syncthreads();
    ring_rows<NW, R>(p, u, t.ub[F]);
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int row = p.row0 + k;
      if (row < p.w) {  // wave-uniform
        const float c = win[k + 5], zm = lane_below(u[k + 1]), zp = lane_above(u[k + 1]), cc = cc_of(rv[k]);
        float v = sponge ? update_coeffs<true, P>(c, prv[k], rv[k], cc, u[k + 1], zm, zp, u[k], u[k + 2],
                                                  sponge_at<P>(damp, t.rows, row))
                         : update_coeffs<false, P>(c, prv[k], rv[k], cc, u[k + 1], zm, zp, u[k], u[k + 2], damp.z);
        if (n > 0 && (SRC || more)) {
          const unsigned h = head.at(k);
          if (h != kNone) v = inject(pt, it & 1, h, chains, !SRC, v);
        }
        if (SRC) {
          grad[k] = grad[k] - v * rc[k] * weight;  // zero-lag imaging condition
          if (band_tile && more && ((inband >> k) & 1)) v = bv[k];
        }
        prv[k] = c;
        if (zin) cur[(row + 6) * LZ + p.lane + 5] = v;
      }
    }
    if (has) pt.amp[(it - 1) & 1][p.tid] = anext;
    if (more) {
      __syncthreads();  // both fields' new edges are in LDS
      // the emptied words have arrived before any word of this step leaves.
      // Both are relaxed stores, so what orders them is this wait and that the
      // hardware acknowledges an agent-scope store only once it is past the
      // L2, where a reader's polls go.  A word whose emptying came late would
      // be taken as data unnoticed (a late stamp of the forward loop is only
      // polled again).  Per word is enough: a word has one writer and one
      // reader thread, the same at every step.
      __builtin_amdgcn_s_waitcnt(0);
      asm volatile("" ::: "memory");
      u64* now = words + turn * copy;
#pragma unroll
      for (int j = 0; j < NE; j++)
        if ((ep.on >> j) & 1) put_pair(&elem(now, ep.q[j]), t.f[0][ep.l[j]], t.f[1][ep.l[j]]);
      if (!collect_pairs<NH>(a.x, now, hp, t.f[0], t.f[1])) t.dead = 1;
      turn = next;
    }
    if (band_tile && more2) {
#pragma unroll
      for (int k = 0; k < R; k++)
        if ((inband >> k) & 1) bv[k] = elem(band + (long long)(it - 2) * a.bsize, bi[k]);
    }
    __syncthreads();
    if (t.dead) return;
  }
  if (SRC) {
    float* out = a.grad + (long long)p.e * a.gstride;
#pragma unroll
    for (int k = 0; k < R; k++)
      if (zin && p.row0 + k < p.w) out[q0 + k * g.ld] = grad[k];
  }
}
template <int P, int R>
__global__ __launch_bounds__(2 * 64 * kResWaves) void k_resident_bwd(ResBwdArgs a) {
  __shared__ BwdTile<P, R> t;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < kResWaves)
    bwd_half<P, R, true>(a, t);
  else
    bwd_half<P, R, false>(a, t);
}

// Calls fn(kernel, threads) with the kernel of a tile width.  Eight waves a
// field, however wide the tile: sixteen with half the rows measured the same
// (301x921 2.65 against 2.67 us a step) or, where some then only wait, worse
// (201x301 2.5 against 1.9).
template <bool BWD, int P, class F>
bool with_width(int w, F&& fn) {
  constexpr int W8 = kResWaves, W16 = 2 * kResWaves;
#define SWFWI_RES_ON(NW, R, KERNEL, THREADS) \
  if (w <= (NW) * (R)) {                     \
    fn(&KERNEL, THREADS);                    \
    return true;                             \
  }
  if constexpr (BWD) {
    SWFWI_RES_ON(W8, 1, (k_resident_bwd<P, 1>), 64 * W16)
    SWFWI_RES_ON(W8, 2, (k_resident_bwd<P, 2>), 64 * W16)
    SWFWI_RES_ON(W8, 3, (k_resident_bwd<P, 3>), 64 * W16)
    SWFWI_RES_ON(W8, 4, (k_resident_bwd<P, 4>), 64 * W16)
    SWFWI_RES_ON(W8, 5, (k_resident_bwd<P, 5>), 64 * W16)
    SWFWI_RES_ON(W8, 6, (k_resident_bwd<P, 6>), 64 * W16)
    SWFWI_RES_ON(W8, 7, (k_resident_bwd<P, 7>), 64 * W16)
    SWFWI_RES_ON(W8, 8, (k_resident_bwd<P, 8>), 64 * W16)
    SWFWI_RES_ON(W8, 9, (k_resident_bwd<P, 9>), 64 * W16)
    SWFWI_RES_ON(W8, 10, (k_resident_bwd<P, 10>), 64 * W16)
  } else {
    SWFWI_RES_ON(W8, 1, (k_resident_fwd<P, 1, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 2, (k_resident_fwd<P, 2, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 3, (k_resident_fwd<P, 3, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 4, (k_resident_fwd<P, 4, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 5, (k_resident_fwd<P, 5, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 6, (k_resident_fwd<P, 6, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 7, (k_resident_fwd<P, 7, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 8, (k_resident_fwd<P, 8, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 10, (k_resident_fwd<P, 10, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 12, (k_resident_fwd<P, 12, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 14, (k_resident_fwd<P, 14, W8>), 64 * W8)
    SWFWI_RES_ON(W8, 16, (k_resident_fwd<P, 16, W8>), 64 * W8)
  }
#undef SWFWI_RES_ON
  return false;
}
template <bool BWD, class F>
bool with_kernel(int precision, int w, F&& fn) {
  return precision == kExact ? with_width<BWD, kExact>(w, fn) : with_width<BWD, kFp32>(w, fn);
}

}  // namespace

int resident_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return cus;
}

int resident_per_cu(bool backward, int precision, int w) {
  int per = 0;
  auto ask = [&](auto k, int threads) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, threads, 0) != hipSuccess) per = 0;
  };
  const bool ok = backward ? with_kernel<true>(precision, w, ask) : with_kernel<false>(precision, w, ask);
  return ok ? per : 0;
}

void launch_resident_fwd(const ResFwdArgs& a, int precision, hipStream_t s) {
  with_kernel<false>(precision, a.g.t.w, [&](auto k, int threads) {
    hipLaunchKernelGGL(k, dim3(a.g.t.n() * a.E), dim3(threads), 0, s, a);
  });
}
void launch_resident_bwd(const ResBwdArgs& a, int precision, hipStream_t s) {
  with_kernel<true>(precision, a.g.t.w, [&](auto k, int threads) {
    hipLaunchKernelGGL(k, dim3(a.g.t.n() * a.E), dim3(threads), 0, s, a);
  });
}

}  // namespace swfwi

// Kernels of the learned coarse-grid correction (learned.h).
//
// One block per 16 x 16 tile of output points (z fastest), 256 threads (4
// waves).  Forward, per tile, every layer on BF16 MFMA with the 16 points of
// a group on the product's N side:
//   stage   p and r p (BF16 pairs) with a 3-cell halo (22 x 22) in LDS;
//   layer 1 D1[c][pt] = sum_k W1^T[c][k] X[k][pt], k = 2 t + (p | r p),
//           over the tile + 2 (20 x 20): two 16x16x16 products (K = 18
//           padded to 32), ReLU, BF16 into LDS;
//   layer 2 D2[co][pt] = sum_t sum_ci W2_t^T[co][ci] h1[ci](pt + o_t) over
//           the tile + 1 (18 x 18): five 16x16x32 products (taps in pairs),
//           ReLU, BF16, kept in registers;
//   layer 3 U[t][pt] = sum_c W3[t][c] h2[c](pt) on the same 18 x 18 points,
//           one 16x16x16 product whose B operand is layer 2's result as it
//           stands (its D layout is the B layout), U into LDS over h1's
//           memory once every wave is past layer 2;
//   output  y(x) = sum_t U[t](x + o_t) on the tile.
// So a 16-point group costs 2 + 5 + 1 products and h2 never leaves the
// registers.
//
// v_mfma_f32_16x16x16_bf16 lane layout (measured on the device): lane l
// supplies A[i = l%16][k = 4*(l/16) + v] and B[k = 4*(l/16) + v][j = l%16]
// as its 4 BF16 items v, and holds D[i = 4*(l/16) + v][j = l%16] in
// accumulator item v.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "learned.h"

namespace swfwi {
namespace {

constexpr int kT = 256;
constexpr int kTile = 16;
// What a block holds around its tile grown by kG cells on every side
template <int kG>
struct Around {
  static constexpr int kP = kTile + 6 + 2 * kG;   // staged field (halo 3)
  static constexpr int kH1 = kTile + 4 + 2 * kG;  // layer-1 region (halo 2)
  static constexpr int kH2 = kTile + 2 + 2 * kG;  // layer-2 region (halo 1)
  static constexpr int kNH1 = kH1 * kH1, kNH2 = kH2 * kH2;
  static constexpr int kGroups1 = kNH1 / 16;         // groups of 16 layer-1 points
  static constexpr int kGroups2 = (kNH2 + 15) / 16;  // and layer-2 points
  static_assert(kNH1 % 16 == 0, "layer-1 points fill whole groups");
};
constexpr int kB = 512;  // threads of the gradient kernel
constexpr int kGrow = 2;  // its outputs reach 2 cells beyond the tile
// Channel pitches of its transposed arrays: layer 1 (a row's point z at z + 2,
// so that the taps of points 4 a .. 4 a + 3 lie in two 8-byte words; 4 channels
// 16 banks apart), dz2 (the same), dz1 (a channel 4 banks on)
constexpr int kH1Pitch = Around<kGrow>::kNH1 + 8, kDz2Pitch = 264, kDz1Pitch = 260;
constexpr int kIn1 = kTile + 2;  // the tile + 1

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 hbf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));

__device__ __host__ __forceinline__ uint16_t bf16_bits(unsigned u) {  // round to nearest even
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ uint16_t bf16_of(float x) { return bf16_bits(__float_as_uint(x)); }
__device__ __forceinline__ float f32_of(uint16_t h) { return __uint_as_float((unsigned)h << 16); }

// accumulator item v of lane l holds D[row][l % 16]
__device__ __forceinline__ int d_row(int l, int v) { return 4 * (l >> 4) + v; }

// (a, b) rounded to BF16 (nearest even) by the hardware conversion
// (v_cvt_pk_bf16_f32), a in the low half; the same bits as bf16_of for
// finite values
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, hbf16x2));
}

// ReLU then BF16 of four accumulator items.  Rounded first, then the
// negative ones (sign bit set: negative as 16-bit integers, -0 included)
// raised to +0 by one packed 16-bit integer max per pair: the same bits as
// rounding max(x, 0).
__device__ __forceinline__ bf16x4 relu_bf16(const f32x4& a) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  const s16x2 zero = {0, 0};
  union { s16x2 h[2]; bf16x4 b; } r;
  r.h[0] = __builtin_elementwise_max(__builtin_bit_cast(s16x2, pack_bf16(a[0], a[1])), zero);
  r.h[1] = __builtin_elementwise_max(__builtin_bit_cast(s16x2, pack_bf16(a[2], a[3])), zero);
  return r.b;
}

// Element i of a field whose base is block-uniform, the byte offset formed in
// 32 bits (a field holds fewer than 2^29 points, checked), so the load takes
// the base from scalar registers and one 32-bit offset
__device__ __forceinline__ float ld_at(const float* base, unsigned i) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + i * 4u);
}

struct TileMap {
  int e, ox, oz;  // entry, tile origin (global padded coords)
  int in;         // the entry's place in the stacks it reads
};

// tiles over the region grown by `margin` cells on every side
__device__ __forceinline__ TileMap tile_of(const NetGeom& g, int margin) {
  const int tz = (g.z1 - g.z0 + 2 * margin + kTile - 1) / kTile, tx = (g.x1 - g.x0 + 2 * margin + kTile - 1) / kTile;
  const int per = tz * tx;
  TileMap m;
  m.e = blockIdx.x / per;
  const int t = blockIdx.x - m.e * per;
  m.ox = g.x0 - margin + (t / tz) * kTile;
  m.oz = g.z0 - margin + (t % tz) * kTile;
  m.in = g.pick ? g.pick[m.e] : m.e;
  return m;
}

// What the gradient keeps of the forward besides (kG > 0)
struct Kept {
  float* in;      // the inputs as the products see them over the tile + 1, [p | r p][kIn1 * kIn1]
  uint16_t* h1t;  // layer 1 channel by channel, [16][kH1Pitch]
  uint16_t* h2;   // layer 2, [point][16]
};

// Shared forward work of a tile grown by kG, by kNT threads.  sx[kP*kP]:
// staged (p, r p) as BF16 pairs (p in the low half); h1[kNH1*16]: layer 1
// (BF16); layer 2 is held in registers and goes through layer 3 into
// u[9][kNH2] (FP32), which may share its memory with h1.  `early` runs among
// the first loads.  Returns false, with nothing computed, when `skip_zero`
// is set and the staged input is zero everywhere (the network, ReLU without
// biases, then gives exactly zero).
template <int kNT, int kG, class Early>
__device__ __forceinline__ bool forward_tile(const float* __restrict__ p, const float* __restrict__ r,
                                             const NetGeom& g, const TileMap& m, const NetDev& w, unsigned* sx,
                                             uint16_t* h1, float* u, bool skip_zero, const Kept& keep, Early early) {
  using A = Around<kG>;
  constexpr int kP = A::kP, kH1 = A::kH1, kH2 = A::kH2, kNH2 = A::kNH2;
  constexpr int kW = kNT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  early();
  int nonzero = 0;
#pragma unroll
  for (int q = tid; q < kP * kP; q += kNT) {
    const int xs = q / kP, zs = q % kP;
    const int x = m.ox - 3 - kG + xs, z = m.oz - 3 - kG + zs;
    const bool in = x >= 0 && x < g.nx && z >= 0 && z < g.nz;
    const unsigned o = (unsigned)(x * g.nz + z);
    const float v = in ? ld_at(p, o) : 0.f;
    const float vq = in ? ld_at(r, o) * v : 0.f;
    const unsigned b = pack_bf16(v, vq);
    sx[q] = b;
    nonzero |= v != 0.f;
    if constexpr (kG > 0) {
      const int xi = xs - 2 - kG, zi = zs - 2 - kG;
      if ((unsigned)xi < (unsigned)kIn1 && (unsigned)zi < (unsigned)kIn1) {
        keep.in[xi * kIn1 + zi] = __uint_as_float(b << 16);
        keep.in[kIn1 * kIn1 + xi * kIn1 + zi] = __uint_as_float(b & 0xffff0000u);
      }
    }
  }
  const int kq = lane >> 4;  // this lane's K quarter
  const bf16x4 a1a = *reinterpret_cast<const bf16x4*>(w.w1a + lane * 4);
  const bf16x4 a1b = *reinterpret_cast<const bf16x4*>(w.w1a + (64 + lane) * 4);
  // layer 2's operands (see there): a block that is the only one of its CU
  // (the gradient's) takes them with the others, as no other's work covers
  // their way from L2; many blocks a CU load them late, for the registers
  hbf16x8 a2p[5];
  auto load_a2p = [&] {
#pragma unroll
    for (int q = 0; q < 5; q++) a2p[q] = *reinterpret_cast<const hbf16x8*>(w.w2p + (q * 64 + lane) * 8);
  };
  if constexpr (kG > 0) load_a2p();
  if (!__syncthreads_or(nonzero) && skip_zero) return false;  // block-uniform
  // layer 1: lane's B items are (p, r p) at taps 2 kq and 2 kq + 1 (first
  // product) and at tap 8 (second product: k = 16 + 4 kq + v, of which only
  // k = 16, 17 have non-zero weights; the other lanes' finite values add
  // exact zeros)
  {
    const int t0 = 2 * kq, t1 = 2 * kq + 1;
    const int o0 = (t0 / 3 - 1) * kP + (t0 % 3 - 1), o1 = (t1 / 3 - 1) * kP + (t1 % 3 - 1);
    const int o8 = kP + 1;
    constexpr int kMaxG1 = (A::kGroups1 + kW - 1) / kW;  // groups per wavefront, at most
#pragma unroll
    for (int i = 0; i < kMaxG1; i++) {
      const int grp = wave + i * kW;
      if (grp >= A::kGroups1) break;  // wave-uniform
      const int q = grp * 16 + (lane & 15);
      const int s = (q / kH1 + 1) * kP + (q % kH1 + 1);  // staged centre
      union { unsigned u2[2]; bf16x4 b; } b0, b1;
      b0.u2[0] = sx[s + o0];
      b0.u2[1] = sx[s + o1];
      b1.u2[0] = sx[s + o8];
      b1.u2[1] = 0u;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1a, b0.b, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1b, b1.b, acc, 0, 0, 0);
      const bf16x4 hv = relu_bf16(acc);
      *reinterpret_cast<bf16x4*>(h1 + q * kNetC + 4 * kq) = hv;  // channels 4 kq .. 4 kq + 3
      if constexpr (kG > 0) {
#pragma unroll
        for (int v = 0; v < 4; v++) keep.h1t[(4 * kq + v) * kH1Pitch + q + 2] = (uint16_t)hv[v];
      }
    }
  }
  __syncthreads();
  // layers 2 and 3
  // five K = 32 products (v_mfma_f32_16x16x32_bf16: lane l supplies
  // A[i = l%16][k = 8*(l/16) + v], B[k = 8*(l/16) + v][j = l%16]): product q
  // takes tap 2q at k < 16 and tap 2q+1 at k >= 16 (channel k%16); the fifth
  // takes tap 8 at k < 16 and zero weights.  One opcode for the whole accumulation
  // chain: a 16x16x16 product that read the accumulator of a 16x16x32 one
  // issued just before it has given wrong sums on gfx950 (no wait states are
  // inserted between the two).
  if constexpr (kG == 0) load_a2p();
  const bf16x4 a3 = *reinterpret_cast<const bf16x4*>(w.w3a + lane * 4);
  const int khalf = kq >> 1, kc = 8 * (kq & 1);  // this lane's tap of the pair, first channel
  // B operand of product q < 4: channels kc .. kc + 7 of tap 2q + khalf of
  // the point's layer-1 neighbourhood; of product 4: those of tap 8 for every
  // lane (the weights past k = 15 are zero and layer-1 values finite, so the
  // lanes of k >= 16 add exact zeros)
  int boff[5];
#pragma unroll
  for (int q = 0; q < 5; q++) {
    const int t = q < 4 ? 2 * q + khalf : 8;
    boff[q] = ((t / 3 - 1) * kH1 + (t % 3 - 1)) * kNetC + kc;
  }
  // layer 2 per group, its result kept in registers; then layer 3 into u:
  // every layer-2 read of h1 is done at the barrier between the two
  constexpr int kMaxG = (A::kGroups2 + kW - 1) / kW;  // groups per wavefront, at most
  bf16x4 hbs[kMaxG];
#pragma unroll
  for (int i = 0; i < kMaxG; i++) {
    const int grp = wave + i * kW;
    if (grp >= A::kGroups2) break;             // wave-uniform
    const int qa = grp * 16 + (lane & 15);     // this lane's point
    const int qs = qa < kNH2 ? qa : kNH2 - 1;  // points past the region read a valid one
    const int x = qs / kH2, z = qs % kH2;      // layer-2 coords; layer-1 = +1
    const uint16_t* c1 = h1 + ((x + 1) * kH1 + (z + 1)) * kNetC;  // the point in layer 1
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const hbf16x8 b = *reinterpret_cast<const hbf16x8*>(c1 + boff[q]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2p[q], b, acc, 0, 0, 0);
    }
    hbs[i] = relu_bf16(acc);  // h2[4 kq + v][qa]
    if constexpr (kG > 0) {
      if (qa < kNH2) *reinterpret_cast<bf16x4*>(keep.h2 + qa * kNetC + 4 * kq) = hbs[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kMaxG; i++) {
    const int grp = wave + i * kW;
    if (grp >= A::kGroups2) break;
    const int qa = grp * 16 + (lane & 15);
    f32x4 y3 = {0.f, 0.f, 0.f, 0.f};
    y3 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a3, hbs[i], y3, 0, 0, 0);  // U[4 kq + v][qa]
    if (qa < kNH2) {
      float* ub = u + 4 * kq * kNH2 + qa;  // row 4 kq; rows past 8 are not kept
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (4 * kq + v < 9) ub[v * kNH2] = y3[v];
    }
  }
  __syncthreads();
  return true;
}

// the output at (x, z) of u's points, of which a row holds kH2
template <int kG>
__device__ __forceinline__ float output_of(const float* u, int x, int z) {
  constexpr int kH2 = Around<kG>::kH2, kNH2 = Around<kG>::kNH2;
  float y = 0.f;
#pragma unroll
  for (int t = 0; t < 9; t++) y += u[t * kNH2 + (x + t / 3 - 1) * kH2 + (z + t % 3 - 1)];
  return y;
}

// 8 waves per SIMD (63 VGPRs, no spills): 5-6% faster than the 7 the
// compiler picks by itself (58 VGPRs plus the accumulators)
__global__ __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(8))) void k_net_apply(
    const float* __restrict__ p_all, float* __restrict__ y_all, NetGeom g, NetDev w) {
  using A = Around<0>;
  __shared__ unsigned sx[A::kP * A::kP];
  // h1 (layer 1) and then u (layer 3): u overwrites h1 after layer 2
  __shared__ __align__(16) uint16_t h1[A::kNH1 * kNetC];
  static_assert(9 * A::kNH2 * sizeof(float) <= A::kNH1 * kNetC * sizeof(uint16_t), "u fits in h1");
  float* u = reinterpret_cast<float*>(h1);
  const TileMap m = tile_of(g, 0);
  const float* p = p_all + (long long)m.in * g.stride;
  const float* r = g.r + (long long)(m.in / g.rdiv) * g.rstride;
  const int x = threadIdx.x / kTile, z = threadIdx.x % kTile;
  const int gx = m.ox + x, gz = m.oz + z;
  float* yo = y_all + (long long)m.e * g.stride + (long long)gx * g.nz + gz;
  const bool out = gx < g.x1 && gz < g.z1;
  if (!forward_tile<kT, 0>(p, r, g, m, w, sx, h1, u, true, Kept{}, [] {})) {
    if (out) *yo = 0.f;
    return;
  }
  if (out) *yo = output_of<0>(u, x + 1, z + 1);
}

__global__ void k_net_add(float* p_all, const float* y_all, NetGeom g) {
  const long long per = (long long)(g.x1 - g.x0) * (g.z1 - g.z0);
  const long long n = per * g.entries;
  for (long long i = blockIdx.x * (long long)kT + threadIdx.x; i < n; i += (long long)gridDim.x * kT) {
    const long long e = i / per, r = i - e * per;
    const int x = g.x0 + (int)(r / (g.z1 - g.z0)), z = g.z0 + (int)(r % (g.z1 - g.z0));
    const long long o = e * g.stride + (long long)x * g.nz + z;
    p_all[o] += y_all[o];
  }
}

// A chain of FP32 products D += a(k, i) b(k, i), batches k = kFrom .. kTo - 1
// of kLen, in order: a batch's operands are read while the one before it is
// multiplied (b BF16, made a float where it is used).  The compiler by itself
// reads each where it is used: 170 cycles a product in place of 70 to 100.
template <int kFrom, int kTo, int kLen, class A, class B>
__device__ __forceinline__ f32x4 mfma_chain(f32x4 acc, A a, B b) {
  float va[2][kLen];
  uint16_t vb[2][kLen];
#pragma unroll
  for (int i = 0; i < kLen; i++) va[0][i] = a(kFrom, i), vb[0][i] = b(kFrom, i);
#pragma unroll
  for (int k = kFrom; k < kTo; k++) {
    const int c = (k - kFrom) & 1, n = c ^ 1;
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1 < kTo) {
#pragma unroll
      for (int i = 0; i < kLen; i++) va[n][i] = a(k + 1, i), vb[n][i] = b(k + 1, i);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kLen; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va[c][i], f32_of(vb[c][i]), acc, 0, 0, 0);
  }
  return acc;
}

// Loss and gradient of one tile.  Forward over the tile + 2, then
//   r = p + net(p) - t, dy = 2 r / count in the region, zero outside it  (tile + 2)
//   dz2[c](x') = relu'(z2) sum_t W3[t][c] dy(x' - o_t)        (tile + 1)
//   dW3[t][c] = sum_tile dy(x) h2[c](x + o_t)                   (FP32 MFMA)
//   dW2[t][ci][co] = sum_tile h1[ci](x + o_t) dz2[co](x)        (BF16 MFMA, K = tile points)
//   dz1[ci](x) = relu'(z1) sum_t sum_co W2[t][ci][co] dz2[co](x - o_t)   (BF16 MFMA)
//   dW1[t][k][c] = sum_tile in_k(x + o_t) dz1[c](x), in_0 = p, in_1 = r p
// into parts[block][kNetParams], the sum of r^2 over the tile into
// lparts[block].  The forward values enter as the forward products saw them:
// inputs, h1, h2 and W3 rounded to BF16; dy and dz1 are FP32 and stay so
// (v_mfma_f32_16x16x4_f32: lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16], D as the others).
//
// A minibatch is about one tile per CU, so the longest chain of one block is
// the kernel's time.  Eight waves share every stage, and the outputs of the
// two cells around the tile, which other blocks hold as well, are computed
// here too: a forward launch and its round trip of dy for a third more
// points.  dW3 is a serial sum over the points of each weight: an FP32
// product of K = 4 adds its four terms to the accumulator one by one in
// order, each a fused multiply-add (measured: the same bits, subnormals
// included), so the wave that walks the points in order gives the bits of
// that sum, and it does so next to the stages of the other waves.  dW1 waits
// for dz1 and is the end of the chain: a thread per weight, whose operands of
// four points come in three reads (LDS-bound, 4200 to 5600 of the block's
// 24000 cycles; 5200 as dependent products on two waves).  dW2's operands
// come channel by channel from transposed copies: three taps from two 8-byte
// reads.
// Measured on 16 samples of 83 x 42 points (288 tiles on 256 CUs): 19.4 us,
// of which a block that has its CU alone takes 11; a forward launch with the
// loss (7.3) and a gradient launch (16.6) before, and with the serial sums on
// four waves 26.7 after 6.5 and 3.0.
__global__ __launch_bounds__(kB) void k_net_grad(const float* __restrict__ p_all, const float* __restrict__ t_all,
                                                 NetGeom g, NetDev w, double inv_count, float* __restrict__ parts,
                                                 double* __restrict__ lparts) {
  using A = Around<kGrow>;
  constexpr int kW = kB / 64, kH1 = A::kH1, kH2 = A::kH2;
  constexpr int kY = kTile + 2 * kGrow;         // dy's points
  constexpr int kN1 = kIn1 * kIn1;              // points of the tile + 1
  static_assert(kY * kY <= kB, "a thread per point of dy");
  __shared__ unsigned sx[A::kP * A::kP];
  __shared__ float in1[2 * kN1];
  __shared__ float sdy[kY * kY];
  // dy over the tile on layer 2's rows, zero around (a row and a point before
  // and after), so that every tap's shift is one offset: the point (x, z) of
  // the tile + 1 at (x + 1) kH2 + z + 1
  constexpr int kTdy = (kIn1 + 2) * kH2;
  __shared__ float tdy[kTdy];
  __shared__ __align__(16) uint16_t h2[A::kNH2 * kNetC];
  __shared__ __align__(16) uint16_t dz2[kN1 * kNetC];         // BF16 (MFMA operand)
  __shared__ __align__(16) uint16_t dz2t[kNetC * kDz2Pitch];  // the tile's own, channel by channel
  __shared__ __align__(16) uint16_t h1t[kNetC * kH1Pitch];
  __shared__ double red[kW];
  __shared__ union __align__(16) {
    uint16_t h1[A::kNH1 * kNetC];    // layer 1 for layer 2,
    float u[9 * A::kNH2];            // then layer 3,
    float dz1[kNetC * kDz1Pitch];    // then dz1, channel by channel
  } mem;
  // tiles cover the region grown by 2: dz2 is non-zero up to 1 and dz1 up
  // to 2 cells outside the region, and every point's terms belong to the
  // one tile that owns it
  const TileMap m = tile_of(g, kGrow);
  const float* p = p_all + (long long)m.in * g.stride;
  const float* tgt = t_all + (long long)m.in * g.stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kq = lane >> 4, ln = lane & 15;
  const int yx = tid / kY, yz = tid % kY;  // this thread's point of dy
  const int gx = m.ox - kGrow + yx, gz = m.oz - kGrow + yz;
  const bool inside = yx < kY && gx >= g.x0 && gx < g.x1 && gz >= g.z0 && gz < g.z1;
  float py = 0.f, ty = 0.f;
  f32x4 w3[9];
  bf16x4 w2[9];
  forward_tile<kB, kGrow>(p, g.r + (long long)(m.in / g.rdiv) * g.rstride, g, m, w, sx, mem.h1, mem.u, false,
                          Kept{in1, h1t, h2}, [&] {
                            if (inside) {
                              py = p[(long long)gx * g.nz + gz];
                              ty = tgt[(long long)gx * g.nz + gz];
                            }
                            // the gradient's operands on their way during the forward
#pragma unroll
                            for (int t = 0; t < 9; t++) {
                              w3[t] = *reinterpret_cast<const f32x4*>(w.w3 + t * kNetC + 4 * kq);
                              w2[t] = *reinterpret_cast<const bf16x4*>(w.w2b + (t * 64 + lane) * 4);
                            }
                            for (int i = tid; i < kTdy; i += kB) tdy[i] = 0.f;
                          });
  {
    double acc = 0;
    if (yx < kY) {
      const int tx = yx - kGrow, tz = yz - kGrow;  // tile coords
      const bool own = (unsigned)tx < (unsigned)kTile && (unsigned)tz < (unsigned)kTile;
      float d = 0.f;
      if (inside) {
        const float res = py + output_of<kGrow>(mem.u, yx + 1, yz + 1) - ty;
        d = (float)(2.0 * res * inv_count);
        if (own) acc = (double)res * res;
      }
      sdy[tid] = d;
      if (own) tdy[(tx + 2) * kH2 + tz + 2] = d;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) red[wave] = acc;
  }
  __syncthreads();
  float* out = parts + (long long)blockIdx.x * kNetParams;
  // dW3, by wave 7 in the time of the others' stages: D[t][c] = sum over the
  // points x' of the tile + 1, in order, of dy(x' - o_t) h2[c](x'), dy taken
  // where x' - o_t is in the tile.  Four points a product, two rows of 18 a
  // batch of nine: item i of lane quarter kq is the pair's point 4 i + kq.
  f32x4 a3 = {0.f, 0.f, 0.f, 0.f};
  const int tl = ln < 9 ? ln : 8;  // the lane's tap; the products' rows past the ninth are not kept
  const float* t3 = tdy + (1 - (tl / 3 - 1)) * kH2 + 1 - (tl % 3 - 1) + kq;
  const uint16_t* b3 = h2 + (kGrow * kH2 + kGrow + kq) * kNetC + ln;
  const int turn = kq < 2 ? 0 : kH2 - kIn1;  // the row ends within item 4
  static_assert(kIn1 == 18, "two rows are nine products");
  const auto at3 = [&](int k, int i) {
    return t3[2 * k * kH2 + 4 * i + (i < 4 ? 0 : i == 4 ? turn : kH2 - kIn1)];
  };
  const auto bt3 = [&](int k, int i) {
    return b3[(2 * k * kH2 + 4 * i + (i < 4 ? 0 : i == 4 ? turn : kH2 - kIn1)) * kNetC];
  };
  constexpr int kCut0 = 3, kCut1 = 7;  // of the nine batches, where the others' stages end
  if (wave == kW - 1) {
    if (lane == 0) {
      double sum = 0;
      for (int i = 0; i < kW; i++) sum += red[i];
      lparts[blockIdx.x] = sum;
    }
    a3 = mfma_chain<0, kCut0, 9>(a3, at3, bt3);
  } else {
    // dz2: lane l has the channels 4 (l / 16) .. + 3 of point l % 16 of a group
    constexpr int kGroups = (kN1 + 15) / 16;
#pragma unroll
    for (int i = 0; i < (kGroups + kW - 2) / (kW - 1); i++) {
      const int q = (wave + i * (kW - 1)) * 16 + ln;
      if (q >= kN1) continue;
      const int x = q / kIn1, z = q % kIn1;  // dy's coords = +1, layer 2's +2
      const bf16x4 hv = *reinterpret_cast<const bf16x4*>(h2 + ((x + kGrow) * kH2 + z + kGrow) * kNetC + 4 * kq);
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 9; t++) {
        const float d = sdy[(x + 1 - (t / 3 - 1)) * kY + (z + 1 - (t % 3 - 1))];
#pragma unroll
        for (int v = 0; v < 4; v++) a[v] = fmaf(w3[t][v], d, a[v]);
      }
      bf16x4 o;
#pragma unroll
      for (int v = 0; v < 4; v++) o[v] = (short)bf16_of(f32_of((uint16_t)hv[v]) > 0.f ? a[v] : 0.f);
      *reinterpret_cast<bf16x4*>(dz2 + q * kNetC + 4 * kq) = o;
      if (x >= 1 && x <= kTile && z >= 1 && z <= kTile) {
#pragma unroll
        for (int v = 0; v < 4; v++) dz2t[(4 * kq + v) * kDz2Pitch + (x - 1) * kTile + z - 1] = (uint16_t)o[v];
      }
    }
  }
  __syncthreads();
  if (wave < 4) {
    // dz1: a row of the tile is a group, D[pt][ci]; two rows at a time
#pragma unroll
    for (int x = wave; x < kTile; x += 8) {
      f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int t = 0; t < 9; t++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const int q2 = (x + 4 * k + 1 - (t / 3 - 1)) * kIn1 + (ln + 1 - (t % 3 - 1));
          const bf16x4 a = *reinterpret_cast<const bf16x4*>(dz2 + q2 * kNetC + 4 * kq);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w2[t], acc[k], 0, 0, 0);
        }
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const uint16_t* h = h1t + ln * kH1Pitch + (x + 4 * k + 2 + kGrow) * kH1 + 4 * kq + 4 + kGrow;
        f32x4 d;
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] = f32_of(h[v]) > 0.f ? acc[k][v] : 0.f;
        *reinterpret_cast<f32x4*>(mem.dz1 + ln * kDz1Pitch + (x + 4 * k) * kTile + 4 * kq) = d;
      }
    }
  } else if (wave < kW - 1) {
    // dW2: waves 4, 5, 6 take a column of taps each; a K-step is a row of the
    // tile, four rows' operands at a time
    const int cx = wave - 5;
    f32x4 a2[3] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    // h1 at z + dz is at 4 kq + (5 .. 7) + v of the row: out of the eight from 4 kq + 4 on
    const uint16_t* ap = h1t + ln * kH1Pitch + (2 + kGrow + cx) * kH1 + 4 * kq + 4;
    const uint16_t* bp = dz2t + ln * kDz2Pitch + 4 * kq;
#pragma unroll
    for (int x0 = 0; x0 < kTile; x0 += 4) {
      uint2 d01[4], d23[4];
      bf16x4 b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        d01[i] = *reinterpret_cast<const uint2*>(ap + (x0 + i) * kH1);
        d23[i] = *reinterpret_cast<const uint2*>(ap + (x0 + i) * kH1 + 4);
        b[i] = *reinterpret_cast<const bf16x4*>(bp + (x0 + i) * kTile);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        union { unsigned u[2]; bf16x4 b; } lo, mid, hi;
        lo.u[0] = __builtin_amdgcn_alignbyte(d01[i].y, d01[i].x, 2);
        lo.u[1] = __builtin_amdgcn_alignbyte(d23[i].x, d01[i].y, 2);
        mid.u[0] = d01[i].y;
        mid.u[1] = d23[i].x;
        hi.u[0] = lo.u[1];
        hi.u[1] = __builtin_amdgcn_alignbyte(d23[i].y, d23[i].x, 2);
        a2[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(lo.b, b[i], a2[0], 0, 0, 0);
        a2[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(mid.b, b[i], a2[1], 0, 0, 0);
        a2[2] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(hi.b, b[i], a2[2], 0, 0, 0);
      }
    }
#pragma unroll
    for (int z = 0; z < 3; z++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        out[kNetW1 + (((cx + 1) * 3 + z) * kNetC + d_row(lane, v)) * kNetC + ln] = a2[z][v];
  } else {
    a3 = mfma_chain<kCut0, kCut1, 9>(a3, at3, bt3);
  }
  __syncthreads();
  if (tid < kNetW1) {
    // dW1: the tile's points in order, a row's operands read while the row
    // before it is added
    const int t = tid / (kNetIn * kNetC), k = (tid / kNetC) % kNetIn, c = tid % kNetC;
    const float* ip = in1 + k * kN1 + (t / 3) * kIn1 + t % 3;
    const float* dp = mem.dz1 + c * kDz1Pitch;
    float vi[2][kTile];
    f32x4 vd[2][kTile / 4];
    auto read = [&](int x) {
#pragma unroll
      for (int z = 0; z < kTile; z++) vi[x & 1][z] = ip[x * kIn1 + z];
#pragma unroll
      for (int z = 0; z < kTile / 4; z++) vd[x & 1][z] = *reinterpret_cast<const f32x4*>(dp + x * kTile + 4 * z);
    };
    float a = 0.f;
    read(0);
#pragma unroll
    for (int x = 0; x < kTile; x++) {
      __builtin_amdgcn_sched_barrier(0);
      if (x + 1 < kTile) read(x + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int z = 0; z < kTile; z++) a = fmaf(vi[x & 1][z], vd[x & 1][z / 4][z % 4], a);
    }
    out[tid] = a;
  }
  if (wave == kW - 1) {
    a3 = mfma_chain<kCut1, 9, 9>(a3, at3, bt3);
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (d_row(lane, v) < 9) out[kNetW1 + kNetW2 + d_row(lane, v) * kNetC + ln] = a3[v];
  }
}

// What k_net_reduce needs to move the weights on as well
struct AdamArgs {
  float *theta, *m, *v;  // theta null: the gradient only
  float c1, c2, lr, b1, b2, eps;
  NetDev w;
};

// weight j's new value into every packed form that holds it (the padding in
// those is zero from k_net_pack on)
__device__ __forceinline__ void pack_weight(const NetDev& w, int j, float th) {
  uint16_t* w1a = const_cast<uint16_t*>(w.w1a);
  uint16_t* w2b = const_cast<uint16_t*>(w.w2b);
  uint16_t* w3a = const_cast<uint16_t*>(w.w3a);
  uint16_t* w2p = const_cast<uint16_t*>(w.w2p);
  const uint16_t b = bf16_of(th);
  if (j < kNetW1) {
    const int k = j / kNetC, c = j % kNetC;
    w1a[(k / 16) * 256 + (((k % 16) / 4) * 16 + c) * 4 + k % 4] = b;
  } else if (j < kNetW1 + kNetW2) {
    const int i = j - kNetW1, t = i / (kNetC * kNetC), ci = (i / kNetC) % kNetC, co = i % kNetC;
    const int k = (t & 1) * 16 + ci;
    w2p[(t / 2) * 512 + ((k / 8) * 16 + co) * 8 + k % 8] = b;
    w2b[t * 256 + ((co / 4) * 16 + ci) * 4 + co % 4] = b;
  } else {
    const int i = j - kNetW1 - kNetW2, t = i / kNetC, c = i % kNetC;
    w3a[((c / 4) * 16 + t) * 4 + c % 4] = b;
    const_cast<float*>(w.w3)[i] = f32_of(b);
  }
}

// grad[j] = sum over blocks of parts[b][j] in FP64, in a fixed order: each
// block takes 16 weights; its 16 thread groups sum consecutive runs of the
// partials in block order, then the 16 run sums are added in run order.  The
// weight's Adam step and its packed forms follow where its gradient is in a
// register, and one more block sums the loss's partials: one launch for what
// four did (288 blocks' partials: 4.8 us in place of 7.0 + 2.4 + 4.2 + 3.1).
constexpr int kRedT = 256, kRedJ = 16, kRedRuns = kRedT / kRedJ;
constexpr int kRedBlocks = (kNetParams + kRedJ - 1) / kRedJ;
__global__ __launch_bounds__(kRedT) void k_net_reduce(const float* __restrict__ parts,
                                                      const double* __restrict__ lparts, long long nblocks,
                                                      float* __restrict__ grad, double* __restrict__ loss, AdamArgs a) {
  __shared__ double run[kRedT];
  if (blockIdx.x == kRedBlocks) {  // the loss: strided sums, then a fixed tree
    double s = 0;
#pragma unroll 4
    for (long long i = threadIdx.x; i < nblocks; i += kRedT) s += lparts[i];
    run[threadIdx.x] = s;
    __syncthreads();
    for (int h = kRedT / 2; h > 0; h >>= 1) {
      if (threadIdx.x < h) run[threadIdx.x] += run[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = run[0];
    return;
  }
  const int jl = threadIdx.x % kRedJ, r = threadIdx.x / kRedJ;
  const int j = blockIdx.x * kRedJ + jl;
  const long long per = (nblocks + kRedRuns - 1) / kRedRuns;
  const long long b0 = r * per, b1 = b0 + per < nblocks ? b0 + per : nblocks;
  double s = 0;
  if (j < kNetParams) {
#pragma unroll 8
    for (long long b = b0; b < b1; b++) s += parts[b * kNetParams + j];
  }
  run[threadIdx.x] = s;
  __syncthreads();
  if (r != 0 || j >= kNetParams) return;
  double t = 0;
#pragma unroll
  for (int q = 0; q < kRedRuns; q++) t += run[q * kRedJ + jl];
  const float gr = (float)t;
  if (grad) grad[j] = gr;
  if (!a.theta) return;
  const float mi = a.b1 * a.m[j] + (1.f - a.b1) * gr;
  const float vi = a.b2 * a.v[j] + (1.f - a.b2) * gr * gr;
  a.m[j] = mi;
  a.v[j] = vi;
  const float th = a.theta[j] - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
  a.theta[j] = th;
  pack_weight(a.w, j, th);
}

__global__ void k_net_pack(const float* theta, uint16_t* w1a, uint16_t* w2b, uint16_t* w3a,
                           uint16_t* w2p, float* w3) {
  const int i = blockIdx.x * kT + threadIdx.x;
  if (i < 5 * 64 * 8) {
    // layer 2, product q: A[co = l%16][k = 8*(l/16) + v] = W2[2q + k/16][k%16][co],
    // zero past tap 8
    const int q = i / 512, l = (i / 8) % 64, v = i % 8;
    const int k = 8 * (l >> 4) + v, co = l & 15, t = 2 * q + (k >> 4);
    w2p[i] = t < 9 ? bf16_of(theta[kNetW1 + (t * kNetC + (k & 15)) * kNetC + co]) : (uint16_t)0;
  }
  if (i < kNetW3) w3[i] = f32_of(bf16_of(theta[kNetW1 + kNetW2 + i]));
  if (i < 2 * 64 * 4) {
    // layer 1, product h: A[c = l%16][k = 16 h + 4*(l/16) + v] = W1 row k (= 2 t + input) or 0 past k = 17
    const int h = i / 256, l = (i / 4) % 64, v = i % 4;
    const int k = 16 * h + 4 * (l >> 4) + v, c = l & 15;
    w1a[i] = k < 9 * kNetIn ? bf16_of(theta[k * kNetC + c]) : (uint16_t)0;
  }
  if (i < 64 * 4) {
    // layer 3: A[t = l%16][c = 4*(l/16) + v] = W3[t][c], rows past tap 8 zero
    const int l = i / 4, v = i % 4;
    const int t = l & 15, c = 4 * (l >> 4) + v;
    w3a[i] = t < 9 ? bf16_of(theta[kNetW1 + kNetW2 + t * kNetC + c]) : (uint16_t)0;
  }
  if (i < 9 * 64 * 4) {
    // item v of lane l for tap t: k = 4*(l/16) + v, n = l%16
    const int t = i / 256, l = (i / 4) % 64, v = i % 4;
    const int k = 4 * (l >> 4) + v, n = l & 15;
    const float* W2 = theta + kNetW1;
    w2b[i] = bf16_of(W2[(t * kNetC + n) * kNetC + k]);  // k = co, n = ci
  }
}

long long tiles_of(const NetGeom& g, int margin) {
  const long long tz = (g.z1 - g.z0 + 2 * margin + kTile - 1) / kTile,
                  tx = (g.x1 - g.x0 + 2 * margin + kTile - 1) / kTile;
  return tz * tx * g.entries;
}

// the staged field reaches 3 cells beyond the tiles, which reach `margin`
// beyond the region
void check_geom(const NetGeom& g, int margin) {
  if (!g.r || g.rdiv < 1) fail(kErrArg, "the network needs the model (1 / vel_t) of every field");
  const int r = 3 + margin;
  if (g.x0 < r || g.z0 < r || g.x1 > g.nx - r || g.z1 > g.nz - r || g.x1 <= g.x0 || g.z1 <= g.z0 || g.entries < 1)
    fail(kErrArg, "network region must lie 5 cells inside the field");
  if (tiles_of(g, margin) > 0x7fffffffLL) fail(kErrRange, "network launch too large");
  if ((long long)g.nx * g.nz >= (1LL << 29)) fail(kErrRange, "network field too large");
}

}  // namespace

void net_pack(const float* theta, const NetDev& w, hipStream_t s) {
  hipLaunchKernelGGL(k_net_pack, dim3((5 * 64 * 8 + kT - 1) / kT), dim3(kT), 0, s, theta, const_cast<uint16_t*>(w.w1a),
                     const_cast<uint16_t*>(w.w2b), const_cast<uint16_t*>(w.w3a),
                     const_cast<uint16_t*>(w.w2p), const_cast<float*>(w.w3));
}

void net_apply(const float* p, float* y, const NetGeom& g, const NetDev& w, hipStream_t s) {
  check_geom(g, 2);
  hipLaunchKernelGGL(k_net_apply, dim3((unsigned)tiles_of(g, 0)), dim3(kT), 0, s, p, y, g, w);
}

void net_add(float* p, const float* y, const NetGeom& g, hipStream_t s) {
  hipLaunchKernelGGL(k_net_add, dim3(2048), dim3(kT), 0, s, p, y, g);
}

long long net_grad_blocks(const NetGeom& g) { return tiles_of(g, kGrow); }

void net_grad(const float* p, const float* t, const NetGeom& g, const NetDev& w, float* parts, double* loss_parts,
              hipStream_t s) {
  check_geom(g, 2);
  const double count = (double)(g.x1 - g.x0) * (g.z1 - g.z0) * g.entries;
  hipLaunchKernelGGL(k_net_grad, dim3((unsigned)tiles_of(g, kGrow)), dim3(kB), 0, s, p, t, g, w, 1.0 / count, parts,
                     loss_parts);
}

void net_reduce(const float* parts, const double* loss_parts, long long nblocks, float* grad, double* loss,
                hipStream_t s) {
  hipLaunchKernelGGL(k_net_reduce, dim3(kRedBlocks + 1), dim3(kRedT), 0, s, parts, loss_parts, nblocks, grad, loss,
                     AdamArgs{});
}

void net_adam(const float* parts, const double* loss_parts, long long nblocks, double* loss, float* theta, float* m,
              float* v, const NetDev& w, int step, float lr, float b1, float b2, float eps, hipStream_t s) {
  const float c1 = 1.f / (1.f - std::pow(b1, (float)step)), c2 = 1.f / (1.f - std::pow(b2, (float)step));
  hipLaunchKernelGGL(k_net_reduce, dim3(kRedBlocks + 1), dim3(kRedT), 0, s, parts, loss_parts, nblocks,
                     (float*)nullptr, loss, AdamArgs{theta, m, v, c1, c2, lr, b1, b2, eps, w});
}

// ---- host handle -------------------------------------------------------------

ConvNet::ConvNet() {
  theta_.resize(kNetParams);
  m_.resize(kNetParams);
  v_.resize(kNetParams);
  grad_.resize(kNetParams);
  w3_.resize(kNetW3);
  w1a_.resize(2 * 64 * 4);
  w2b_.resize(9 * 64 * 4);
  w3a_.resize(64 * 4);
  w2p_.resize(5 * 64 * 8);
  lsum_.resize(1);
}

void ConvNet::repack(hipStream_t s) { net_pack(theta_.get(), dev(), s); }

void ConvNet::set_weights(const float* host) {
  SWFWI_HIP(hipMemcpy(theta_.get(), host, sizeof(float) * kNetParams, hipMemcpyHostToDevice));
  SWFWI_HIP(hipMemset(m_.get(), 0, sizeof(float) * kNetParams));
  SWFWI_HIP(hipMemset(v_.get(), 0, sizeof(float) * kNetParams));
  step_ = 0;
  repack(nullptr);
  SWFWI_HIP(hipDeviceSynchronize());
}

void ConvNet::get_weights(float* host) const {
  SWFWI_HIP(hipMemcpy(host, theta_.get(), sizeof(float) * kNetParams, hipMemcpyDeviceToHost));
}

void ConvNet::correct(float* p, const NetGeom& g, float* yscratch, hipStream_t s) const {
  net_apply(p, yscratch, g, dev(), s);
  net_add(p, yscratch, g, s);
}

// the blocks' gradients and losses
void ConvNet::grad_parts(const float* in, const float* target, const NetGeom& g, hipStream_t s) {
  parts_.resize((size_t)net_grad_blocks(g) * kNetParams);
  lparts_.resize((size_t)net_grad_blocks(g));
  net_grad(in, target, g, dev(), parts_.get(), lparts_.get(), s);
}

double ConvNet::loss_grad(const float* in, const float* target, const NetGeom& g, float* grad_host, hipStream_t s) {
  grad_parts(in, target, g, s);
  net_reduce(parts_.get(), lparts_.get(), net_grad_blocks(g), grad_.get(), lsum_.get(), s);
  double loss = 0;
  SWFWI_HIP(hipMemcpyAsync(&loss, lsum_.get(), sizeof(double), hipMemcpyDeviceToHost, s));
  if (grad_host) SWFWI_HIP(hipMemcpyAsync(grad_host, grad_.get(), sizeof(float) * kNetParams, hipMemcpyDeviceToHost, s));
  SWFWI_HIP(hipStreamSynchronize(s));
  const double count = (double)(g.x1 - g.x0) * (g.z1 - g.z0) * g.entries;
  return loss / count;
}

void ConvNet::train_step(const float* in, const float* target, const NetGeom& g, float lr, double* loss_dev,
                         hipStream_t s) {
  grad_parts(in, target, g, s);
  step_++;
  net_adam(parts_.get(), lparts_.get(), net_grad_blocks(g), loss_dev, theta_.get(), m_.get(), v_.get(), dev(), step_,
           lr, 0.9f, 0.999f, 1e-8f, s);
}

void ConvNet::set_data(const float* in_host, const float* r_host, const float* target_host, int n,
                       const NetGeom& g) {
  if (n < 1) fail(kErrArg, "empty training set");
  dg_ = g;
  dg_.entries = 1;
  dg_.stride = (long long)g.nx * g.nz;
  dn_ = n;
  const size_t len = (size_t)n * dg_.stride;
  din_.resize(len);
  dr_.resize(len);
  dtgt_.resize(len);
  SWFWI_HIP(hipMemcpy(din_.get(), in_host, sizeof(float) * len, hipMemcpyHostToDevice));
  SWFWI_HIP(hipMemcpy(dr_.get(), r_host, sizeof(float) * len, hipMemcpyHostToDevice));
  SWFWI_HIP(hipMemcpy(dtgt_.get(), target_host, sizeof(float) * len, hipMemcpyHostToDevice));
}

void ConvNet::train(int batch, int steps, float lr, unsigned long long seed, double* losses, hipStream_t s) {
  if (!dn_) fail(kErrState, "no training set");
  if (batch < 1 || batch > dn_) fail(kErrArg, "minibatch size out of range");
  if (steps < 0) fail(kErrArg, "negative step count");
  NetGeom g = dg_;
  g.entries = batch;
  g.r = dr_.get();
  g.rstride = g.stride;
  g.rdiv = 1;
  // seeded shuffle of the sample order (splitmix64 + Fisher-Yates), refreshed
  // each pass; the minibatch of step k is idx[k * batch .. (k + 1) * batch)
  std::vector<int> order(dn_), idx((size_t)steps * batch);
  for (int i = 0; i < dn_; i++) order[i] = i;
  unsigned long long st = seed;
  auto next = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    unsigned long long z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  int pos = dn_;
  for (size_t q = 0; q < idx.size(); q++) {
    if (pos == dn_) {
      for (int i = dn_ - 1; i > 0; i--) std::swap(order[i], order[(int)(next() % (unsigned long long)(i + 1))]);
      pos = 0;
    }
    idx[q] = order[pos++];
  }
  if (steps == 0) return;
  DBuf<int> didx;
  DBuf<double> dloss;
  didx.upload(idx.data(), idx.size(), s);
  dloss.resize((size_t)steps);
  for (int k = 0; k < steps; k++) {
    g.pick = didx.get() + (size_t)k * batch;
    train_step(din_.get(), dtgt_.get(), g, lr, dloss.get() + k, s);
  }
  std::vector<double> l((size_t)steps);
  dloss.download(l.data(), l.size(), s);
  SWFWI_HIP(hipStreamSynchronize(s));
  const double count = (double)(g.x1 - g.x0) * (g.z1 - g.z0) * g.entries;
  if (losses)
    for (int k = 0; k < steps; k++) losses[k] = l[k] / count;
}

}  // namespace swfwi

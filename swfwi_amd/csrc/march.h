// What the strip-walking step kernels share: a wave owns a strip of up to 128
// consecutive z, two per lane, and walks it along x with a ring of rows in
// registers and a row buffer of its own in LDS.
#pragma once
#include <hip/hip_runtime.h>

namespace swfwi {
namespace march {

constexpr int kWaves = 4;             // waves of a block, each on its own
constexpr int kRing = 16;             // rows of cur in registers: 11 of the stencil, 5 ahead
constexpr int kAhead = 4;             // rows that prev and the model are loaded ahead (8: no faster)
constexpr int kRowPad = 8;            // LDS floats before and after a row buffer
constexpr int kRowLen = 128 + 2 * kRowPad;

typedef float f2 __attribute__((ext_vector_type(2)));

// An array of an entry as a buffer: its base and size in four scalar registers,
// so that an access takes a row's byte offset (scalar) and a lane's (vector) as
// they are, with no address arithmetic, and one past the end reads 0.
typedef __amdgpu_buffer_rsrc_t Buf;
__device__ __forceinline__ Buf buffer_of(const void* p, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (unsigned)bytes, 0x00020000);
}
typedef unsigned u2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f2 load2(Buf b, unsigned lane_bytes, unsigned row_bytes) {
  return __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(b, lane_bytes, row_bytes, 0));
}
__device__ __forceinline__ void store2(Buf b, unsigned lane_bytes, unsigned row_bytes, f2 v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, v), b, lane_bytes, row_bytes, 0);
}
__device__ __forceinline__ void store1(Buf b, unsigned lane_bytes, unsigned row_bytes, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), b, lane_bytes, row_bytes, 0);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// the second element of the lane below, the first of the lane above
__device__ __forceinline__ float below(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float above(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}

// z neighbours of a lane's two elements in a row: n[0..4] = z-5..z-1 of the
// first, n[5..9] = z+1..z+5 of the second.
template <int R>
struct Zn {
  float lo[R], hi[R];
};
template <int R>
__device__ __forceinline__ Zn<R> z_neighbours(const float* row, int lane) {
  const float* p = row + kRowPad + 2 * lane;
  Zn<R> n;
#pragma unroll
  for (int k = 0; k < R; k++) {
    n.lo[k] = p[-1 - k];
    n.hi[k] = p[2 + k];
  }
  return n;
}

}  // namespace march
}  // namespace swfwi

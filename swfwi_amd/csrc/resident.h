// Resident time loop: a whole forward or backward run of a small batch as ONE
// launch whose blocks keep their tiles on chip and trade halos through memory.
//
// A batch whose fields fit the chip's registers and LDS (one supershot, the
// line search's trials, a few small shots) is not bound by bandwidth but by
// the chain launch -> load -> LDS -> store of every step (about 5 us).  Here
// block b owns one tile of one entry for all steps: prev, model and gradient
// live in registers, cur with its 6-cell halo in LDS, and per step a block
// only publishes the 6-wide edge of its new field and collects its neighbours'
// edges.
//
// Exchange: a published value travels as one 8-byte word (value, stamp), the
// two fields' values of the backward loop as one word that is empty before,
// written and read with relaxed agent-scope atomics (single-copy atomic, past
// the per-XCD L2s), so a reader knows a value has arrived from the word
// itself: no flags, fences or cache write-backs.  Stamps grow over the life of
// the buffer, so nothing has to be cleared between runs; two copies alternate
// by step parity.  A block publishes step t+2 over its step t only after it
// has collected step t+1 from every tile that reads it, and those published
// t+1 after their block had collected t: nothing is overwritten unread.
//
// Waits are bounded: a block that waits longer than the limit raises an abort
// flag that every waiting block polls, all blocks then leave, and the caller
// runs the per-step kernels instead.  The launch needs every block on the chip
// at once; the host checks the blocks against the device's capacity and lets
// one resident run at a time onto a device.  A batch that does not fit goes as
// a few launches of a part of its entries each, over one buffer.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "kernels.h"

namespace swfwi {

constexpr int kResWaves = 8;                // waves of a field (the forward kernel has one, the backward two)
constexpr int kResTileZ = 62;               // most outputs along z: lanes 1..62, lanes 0 and 63 the u2 ring
constexpr int kResLdz = 64 + 2 * 6;         // LDS row of a tile: z from -6 to 69
constexpr int kResMaxPts = 512;             // sources or receivers of one tile, one per thread
constexpr int kResMaxWidthFwd = 128;        // widest tile (x)
constexpr int kResMaxWidthBwd = 80;          // (spills from 57 columns on; 69 columns still 9.1 against 11.4 us per step)
constexpr int kResLanesRows = 8, kResLanesRows2 = 5;  // most rows a wave for 2 to 4 forward entries, one block a CU and two
constexpr int kResTwiceRows = 6;             // most rows a wave of which two forward blocks fit a CU

// Fewest steps of a resident run: its launch, wait and clears cost about 10 us
// (whole calls of one shot on 201x301 / 501x1501, launches -> resident: 2 steps
// 82 -> 91 / 85 -> 104 us, 3 steps 82 -> 91 / 90 -> 105, 5 steps 107 -> 93 / 118 ->
// 115, 10 steps 127 -> 103 / 147 -> 133).
constexpr int kResSteps = 5;
constexpr int kResMaxPartsFwd = 3, kResMaxPartsBwd = 8;  // most launches of one run
constexpr int kResWideFwd = 15, kResWideBwd = 10;  // rows a wave from which parts are faster than one launch
constexpr int kResPartRows = 7;               // most rows a wave of a part
constexpr double kResWideUs[2] = {8.6, 7.5};  // a forward step of kResWideFwd rows and more, exact and FP32
constexpr double kResPartUs = 20;             // a part's launch and clears

// Tiles of one entry: w x h outputs each (the last column and row may be smaller).
struct ResTiles {
  int ntx = 0, ntz = 0, w = 0, h = 0;
  int n() const { return ntx * ntz; }
};

// Sources or receivers by tile: items [ptr[t], ptr[t+1]) are (row << 6 | lane,
// point id) in ascending id.
struct ResPoints {
  const int* ptr = nullptr;
  const int2* items = nullptr;
};

struct ResComm {
  unsigned long long* buf = nullptr;  // forward [2][E][npts] stamped words, backward [3][E][npts] pairs, empty
  unsigned base = 0;                  // stamps of a forward run are base + 1 ...
  int* abort_dev = nullptr;           // set by a block that gives up
  int* abort_host = nullptr;          // the same for the host (mapped)
  long long limit = 0;                // longest wait, in 100 MHz ticks
};

struct ResGrid {
  int nx = 0, nz = 0, ld = 0;
  int nb = 0, zdamp = 0;
  int bx0 = 0, bxn = 0, bz0 = 0, bzn = 0;
  const float* delta_x = nullptr;
  const float* delta_z = nullptr;
  ResTiles t;
  int e0 = 0;  // the launch takes the entries from here on; the exchange counts from it
};

struct ResFwdArgs {
  ResGrid g;
  ResComm x;
  int E = 1, nt = 0;  // (E: entries of this launch)
  long long fstride = 0;
  float* fa = nullptr;  // in: p(-1); the two then hold p(nt-1) and p(nt) as the per-step loop leaves them
  float* fb = nullptr;  // in: p(0)
  const float* rv = nullptr;
  long long rvstride = 0;
  int rvdiv = 1;
  ResPoints src, rec;
  const float* amp = nullptr;
  int amp_ld = 0;
  long long amp_estride = 0;
  const int *lo = nullptr, *hi = nullptr;
  float* dcal = nullptr;
  int ng = 0;
  float* band = nullptr;
  int bsize = 0;
};

struct ResBwdArgs {
  ResGrid g;
  ResComm x;
  int E = 1, nt = 0, it_min = 0;
  long long fstride = 0;
  const float* s_cur = nullptr;  // p(nt-1)
  const float* s_nxt = nullptr;  // p(nt)
  const float* g_cur = nullptr;  // the receiver field with the last sample injected
  const float* rv = nullptr;
  long long rvstride = 0;
  int rvdiv = 1;
  ResPoints src, rec;
  const float* amp = nullptr;
  int amp_ld = 0;
  long long amp_estride = 0;
  const int *lo = nullptr, *hi = nullptr;
  const float* vsrc = nullptr;
  int ng = 0;
  long long vstride = 0;
  const float* band = nullptr;
  int bsize = 0;
  const float* weights = nullptr;  // [nt]
  float* grad = nullptr;           // written (interior points)
  long long gstride = 0;
};

// CUs of the device, and blocks of the kernel for tile width w that fit one at once (0: none).
int resident_cus();
int resident_per_cu(bool backward, int precision, int w);
void launch_resident_fwd(const ResFwdArgs& a, int precision, hipStream_t s);
void launch_resident_bwd(const ResBwdArgs& a, int precision, hipStream_t s);

}  // namespace swfwi

// Small kernels around the mixed-size batch's time loops (batch.h): the step-0
// injections, the residual and the fills.
#include <hip/hip_runtime.h>

#include "batch.h"
#include "kernels.h"

namespace swfwi {
namespace {

constexpr int kBT = 256;
// step-0 fields: both buffers zero (by the caller), then the first source
// amplitude (forward) or the last adjoint-source sample (backward) in fb
__global__ void k_batch_inject0(BatchKernelArgs a, int nentries, int fwd) {
  const int e = blockIdx.x;
  if (e >= nentries) return;
  const BatchEntry E = a.ent[e];
  if (fwd) {
    if (threadIdx.x == 0) a.fb[E.f + E.src] = a.amp[E.amp0];
  } else {
    const int ld = E.nzpad;
    for (int r = threadIdx.x; r < E.ng; r += blockDim.x)
      a.fb[E.f + E.rec0 + (long long)r * ld] = a.dcal[E.dcal + (long long)(E.nt - 1) * E.ng + r];
  }
}

__global__ void k_sub(const float* a, const float* b, float* out, long long n) {
  for (long long i = blockIdx.x * (long long)kBT + threadIdx.x; i < n; i += (long long)gridDim.x * kBT)
    out[i] = a[i] - b[i];
}

__global__ void k_fill_u32(unsigned* p, long long n, unsigned v) {
  for (long long i = blockIdx.x * (long long)kBT + threadIdx.x; i < n; i += (long long)gridDim.x * kBT) p[i] = v;
}

}  // namespace

void launch_fill_u32(unsigned* p, long long n, unsigned v, hipStream_t s) {
  long long b = (n + kBT - 1) / kBT;
  if (b > 4096) b = 4096;
  if (b < 1) b = 1;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)b), dim3(kBT), 0, s, p, n, v);
}

void launch_sub(const float* a, const float* b, float* out, long long n, hipStream_t s) {
  long long blk = (n + kBT - 1) / kBT;
  if (blk > 8192) blk = 8192;
  if (blk < 1) blk = 1;
  hipLaunchKernelGGL(k_sub, dim3((unsigned)blk), dim3(kBT), 0, s, a, b, out, n);
}

void launch_batch_init_fwd(const BatchKernelArgs& a, int nentries, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_inject0, dim3(nentries), dim3(64), 0, s, a, nentries, 1);
}
void launch_batch_init_bwd(const BatchKernelArgs& a, int nentries, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_inject0, dim3(nentries), dim3(kBT), 0, s, a, nentries, 0);
}

}  // namespace swfwi

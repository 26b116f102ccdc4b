// Launches of the F-stage of 1024 real points (fstage_1k.hpp).
#include "fstage_1k.hpp"

namespace gxc {
namespace {

using namespace fs;
using one::fstage_1k_item;
using one::kBytes;

template <int OUT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) fstage_1k_kernel(FParams p) {
  __shared__ __align__(16) unsigned char smem[kBytes];
  fstage_1k_item<OUT>(p, (int)xcd_order(blockIdx.x, gridDim.x), smem);  // grid = nant * nt exactly
}

// Several subbands: unit = item.
template <int OUT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
fstage_1k_group_kernel(const FSeg *__restrict__ segs, int nseg) {
  __shared__ __align__(16) unsigned char smem[kBytes];
  const long long u = xcd_order(blockIdx.x, gridDim.x);
  const int k = find_fseg(segs, nseg, u);
  const FParams p = segment_params(segs, k);
  fstage_1k_item<OUT>(p, (int)(u - segs[k].unit0), smem);
}

}  // namespace

hipError_t launch_fstage_1k(const FParams &p, hipStream_t s) {
  const long long items = (long long)p.nant * p.nt;
  if (items <= 0) return hipSuccess;
  if (items > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)items), block(64);
  switch (p.out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_1k_kernel<OUT_F32>), grid, block, 0, s, p); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_1k_kernel<OUT_F16>), grid, block, 0, s, p); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_1k_kernel<OUT_BF16>), grid, block, 0, s, p); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_1k_kernel<OUT_FP8>), grid, block, 0, s, p); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_1k_kernel<OUT_POWER>), grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_fstage_1k_group(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s) {
  const dim3 grid((unsigned)units), block(64);
  switch (out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_1k_group_kernel<OUT_F32>), grid, block, 0, s, segs, nseg); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_1k_group_kernel<OUT_F16>), grid, block, 0, s, segs, nseg); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_1k_group_kernel<OUT_BF16>), grid, block, 0, s, segs, nseg); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_1k_group_kernel<OUT_FP8>), grid, block, 0, s, segs, nseg); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_1k_group_kernel<OUT_POWER>), grid, block, 0, s, segs, nseg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace gxc

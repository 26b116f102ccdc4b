// The F-stage of a batch's short subbands of several FFT lengths in one launch: a
// workgroup of 256 threads takes one unit of its subband's length, real input.
// Launches by length cost about 6 us each where none fills the chip.  Here every
// workgroup holds the registers and LDS of the longest length, four to a CU, and
// has idle waves from 1024 to 4096 points, about 3 us per 1000 units of those:
// hence 1500 units per launch saved (kFMixedUnits).  Whole passes in us, by length
// -> together: 4 stations, 4 subbands of 128 .. 1024 channels x 100 FFTs (450
// units) FP32 73 -> 52, FP16 118 -> 85; 3 stations, 8 subbands of 256 .. 4096
// channels, 1 ms (990) 117 -> 77, 176 -> 116; the same of 6 ms (5913 units, 5
// lengths) 165 -> 157, 227 -> 188; past the line, 512 channels x 1000 and 1024 x
// 500 (6000 units, 2 lengths) 87 -> 98.
#include "fstage16.hpp"
#include "fstage_1k.hpp"
#include "fstage_big.hpp"

namespace gxc {
namespace {

using namespace fs;

// Segment and unit come by opaque copies, and an end of its own, so that no
// code is shared with the other lengths: what is moved out of a length's code
// rounds differently there, and the spectra are to be those of the launches by
// length, bit for bit.
template <int L, int OUT>
__device__ __forceinline__ void mixed_item(const FSeg *__restrict__ segs, int k, unsigned char *smem) {
  constexpr int T = L < 1024 ? 256 : L == 1024 ? 64 : L / 32;
  // whole waves leave here, and a barrier waits for those that are left
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= T / 64) return;
  asm volatile("; %1 points" : "+s"(k) : "n"(L));
  const FParams p = segment_params(segs, k);
  const int unit = blockIdx.x - (int)segs[k].unit0;
  if constexpr (L < 1024)
    fstage16_item<L, false, OUT, 2048 / L>(p, unit, smem);
  else if constexpr (L == 1024)
    one::fstage_1k_item<OUT>(p, unit, smem);
  else
    fstage_big_item<L, false, OUT, true>(p, unit, smem);
  asm volatile("; %0 points" ::"n"(L) : "memory");
}

constexpr int kLds = std::max({QLds<256, false, 8>::BYTES, QLds<512, false, 4>::BYTES, one::kBytes,
                               BLds<2048, false>::BYTES, BLds<4096, false>::BYTES, BLds<8192, false>::BYTES});

template <int OUT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
fstage_mixed_kernel(const FSeg *__restrict__ segs, int nseg) {
  __shared__ __align__(16) unsigned char smem[kLds];
  const int k = find_fseg(segs, nseg, blockIdx.x);
  switch (__builtin_amdgcn_readfirstlane(segs[k].L)) {
    case 256: mixed_item<256, OUT>(segs, k, smem); break;
    case 512: mixed_item<512, OUT>(segs, k, smem); break;
    case 1024: mixed_item<1024, OUT>(segs, k, smem); break;
    case 2048: mixed_item<2048, OUT>(segs, k, smem); break;
    case 4096: mixed_item<4096, OUT>(segs, k, smem); break;
    default: mixed_item<8192, OUT>(segs, k, smem); break;
  }
}

}  // namespace

hipError_t launch_fstage_mixed(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s) {
  const dim3 grid((unsigned)units), block(256);
  switch (out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_mixed_kernel<OUT_F32>), grid, block, 0, s, segs, nseg); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_mixed_kernel<OUT_F16>), grid, block, 0, s, segs, nseg); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_mixed_kernel<OUT_BF16>), grid, block, 0, s, segs, nseg); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_mixed_kernel<OUT_FP8>), grid, block, 0, s, segs, nseg); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_mixed_kernel<OUT_POWER>), grid, block, 0, s, segs, nseg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace gxc

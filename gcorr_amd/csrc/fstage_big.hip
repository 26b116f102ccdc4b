// Per-subband launch of the F-stage of 2048 points and more (fstage_big.hpp):
// one workgroup of L/32 threads per (station, FFT) for real input up to 8192
// points, per (station, FFT, pol) otherwise.
#include "fstage_big.hpp"

namespace gxc {
namespace {

using namespace fs;

// For real input up to 8192 points a workgroup takes both polarisations of
// one (station, FFT) in turn, so the delay split, the rotator tables and the
// pass-0 matrix are built once for two FFTs.  Above, one polarisation is
// already 512 and 1024 threads, and complex input would hold 32 registers of
// M's operands over the first FFT.
template <int L, bool CPLX>
constexpr bool big_both() { return !CPLX && L <= 8192; }

template <int L, bool CPLX, int OUT>
__global__ void __launch_bounds__((BG<L, CPLX>::T)) __attribute__((amdgpu_waves_per_eu(4)))
fstage_big_kernel(FParams p) {
  __shared__ __align__(16) unsigned char smem[BLds<L, CPLX>::BYTES];
  // grid = nant * nt (both polarisations per workgroup) or 2 * nant * nt
  // exactly; in the second form the two polarisations of one (station,
  // FFT) are consecutive units on one XCD, so the second finds the input
  // words in L2
  fstage_big_item<L, CPLX, OUT, big_both<L, CPLX>()>(p, (int)xcd_order(blockIdx.x, gridDim.x), smem);
}

// Several subbands, real input: unit = item, both polarisations.
template <int L, int OUT>
__global__ void __launch_bounds__((BG<L, false>::T)) __attribute__((amdgpu_waves_per_eu(4)))
fstage_big_group_kernel(const FSeg *__restrict__ segs, int nseg) {
  static_assert(big_both<L, false>(), "unit = item");
  __shared__ __align__(16) unsigned char smem[BLds<L, false>::BYTES];
  const long long u = xcd_order(blockIdx.x, gridDim.x);
  const int k = find_fseg(segs, nseg, u);
  const FParams p = segment_params(segs, k);
  fstage_big_item<L, false, OUT, true>(p, (int)(u - segs[k].unit0), smem);
}

template <int L>
hipError_t launch_group(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s) {
  const dim3 grid((unsigned)units), block(BG<L, false>::T);
  switch (out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_big_group_kernel<L, OUT_F32>), grid, block, 0, s, segs, nseg); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_big_group_kernel<L, OUT_F16>), grid, block, 0, s, segs, nseg); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_big_group_kernel<L, OUT_BF16>), grid, block, 0, s, segs, nseg); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_big_group_kernel<L, OUT_FP8>), grid, block, 0, s, segs, nseg); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_big_group_kernel<L, OUT_POWER>), grid, block, 0, s, segs, nseg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int L, bool CPLX>
hipError_t launch_big(const FParams &p, hipStream_t s) {
  using G = BG<L, CPLX>;
  const long long items = (big_both<L, CPLX>() ? 1LL : 2LL) * p.nant * p.nt;
  if (items <= 0) return hipSuccess;
  if (items > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)items), block(G::T);
  switch (p.out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_big_kernel<L, CPLX, OUT_F32>), grid, block, 0, s, p); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_big_kernel<L, CPLX, OUT_F16>), grid, block, 0, s, p); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_big_kernel<L, CPLX, OUT_BF16>), grid, block, 0, s, p); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_big_kernel<L, CPLX, OUT_FP8>), grid, block, 0, s, p); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_big_kernel<L, CPLX, OUT_POWER>), grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fstage_big(const FParams &p, int L, bool cplx, hipStream_t s) {
  switch (L) {
    case 2048: return cplx ? launch_big<2048, true>(p, s) : launch_big<2048, false>(p, s);
    case 4096: return cplx ? launch_big<4096, true>(p, s) : launch_big<4096, false>(p, s);
    case 8192: return cplx ? launch_big<8192, true>(p, s) : launch_big<8192, false>(p, s);
    case 16384: return cplx ? launch_big<16384, true>(p, s) : launch_big<16384, false>(p, s);
    case 32768: return cplx ? launch_big<32768, true>(p, s) : launch_big<32768, false>(p, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_fstage_big_group(const FSeg *segs, int nseg, long long units, int L, int out_mode, hipStream_t s) {
  switch (L) {
    case 2048: return launch_group<2048>(segs, nseg, units, out_mode, s);
    case 4096: return launch_group<4096>(segs, nseg, units, out_mode, s);
    case 8192: return launch_group<8192>(segs, nseg, units, out_mode, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gxc

// Multi-subband F-stage: the subbands of 256..1024 points of a subintegration
// in one persistent launch.  Subbands differ in FFT length, bandwidth, delays and input; the
// workgroup size is common, so a unit of work is one workgroup's worth of
// items (station, FFT) of one subband.  Units are strided over a grid sized
// to fill the device once; each unit runs the same item code as the
// per-subband launch (fstage16.hpp).
#include "fstage16.hpp"

namespace gxc {
namespace {

using namespace fs;

// Workgroups of 256 threads: 2048 / L items with both polarisations.
constexpr int kBlock = 256;
constexpr int m_ipw(int L) { return kBlock / (L / 8); }
constexpr int max2(int a, int b) { return a > b ? a : b; }
constexpr int kMultiLds = max2(max2(QLds<256, false, m_ipw(256)>::BYTES, QLds<512, false, m_ipw(512)>::BYTES),
                               QLds<1024, false, m_ipw(1024)>::BYTES);

// One unit at FFT length L, kept out of line: each length gets its own
// register allocation instead of one merged over every length.
template <int L, int OUT>
__device__ __attribute__((noinline)) void multi_unit(const FSeg *g, int blk, unsigned char *smem) {
  fstage16_item<L, false, OUT, m_ipw(L)>(g->p, blk, smem);
}

template <int OUT>
__global__ void __launch_bounds__(kBlock) fstage_multi_kernel(const FSeg *segs, int nseg, long long total) {
  __shared__ __align__(16) unsigned char smem[kMultiLds];
  // Units in plain order: their cost differs by subband (FFT length), and
  // striding them over the grid spreads every subband over every XCD.
  for (long long u = blockIdx.x; u < total; u += gridDim.x) {
    int k = 0;
    while (k + 1 < nseg && u >= segs[k + 1].unit0) ++k;
    const FSeg &g = segs[k];
    const int blk = (int)(u - g.unit0);
    __syncthreads();  // the previous unit's LDS reads are done
    switch (g.L) {
      case 256: multi_unit<256, OUT>(&g, blk, smem); break;
      case 512: multi_unit<512, OUT>(&g, blk, smem); break;
      case 1024: multi_unit<1024, OUT>(&g, blk, smem); break;
    }
  }
}

}  // namespace

int fstage_multi_block() { return kBlock; }

long long fstage_multi_units(int L, long long items) {
  const long long ipw = m_ipw(L);
  return (items + ipw - 1) / ipw;
}

hipError_t launch_fstage_multi(const FSeg *segs, int nseg, long long total, int out_mode, hipStream_t s) {
  if (total <= 0) return hipSuccess;
  const void *fn = nullptr;
  switch (out_mode) {
    case OUT_F32: fn = reinterpret_cast<const void *>(&fstage_multi_kernel<OUT_F32>); break;
    case OUT_F16: fn = reinterpret_cast<const void *>(&fstage_multi_kernel<OUT_F16>); break;
    case OUT_BF16: fn = reinterpret_cast<const void *>(&fstage_multi_kernel<OUT_BF16>); break;
    case OUT_FP8: fn = reinterpret_cast<const void *>(&fstage_multi_kernel<OUT_FP8>); break;
    case OUT_POWER: fn = reinterpret_cast<const void *>(&fstage_multi_kernel<OUT_POWER>); break;
    default: return hipErrorInvalidValue;
  }
  const long long grid = persistent_grid(fn, kBlock, 0, total);
  void *args[] = {(void *)&segs, (void *)&nseg, (void *)&total};
  return hipLaunchKernel(fn, dim3((unsigned)grid), dim3(kBlock), args, 0, s);
}

}  // namespace gxc

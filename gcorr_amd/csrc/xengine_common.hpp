// Device helpers shared by the X-stage kernels: xengine.hip (the general form)
// and xsplit.hip (the streaming form: FP16 and BF16 spectra of up to 32 inputs,
// FP32 spectra of the F-stage).
#pragma once

#include "gxc_xengine.hpp"

namespace gxc {
namespace xs {

// sum + comp += v with Neumaier's compensation (the rounding error of each
// addition kept in comp).
__device__ __forceinline__ void neumaier(float &sum, float &comp, float v) {
#pragma clang fp contract(off)
  const float t = sum + v;
  if (fabsf(sum) >= fabsf(v))
    comp += (sum - t) + v;
  else
    comp += (v - t) + sum;
  sum = t;
}

// One value of this chunk into element e of a partial plane.  With a
// compensation plane (subintegrations of several chunks) each later chunk is
// added with Neumaier's compensation, the first clears it.
__device__ __forceinline__ void put_partial(bool accumulate, float *pl, float *cpl, size_t e, float v) {
  if (!accumulate) {
    pl[e] = v;
    if (cpl) cpl[e] = 0.f;
  } else if (cpl) {
    float sum = pl[e], comp = cpl[e];
    neumaier(sum, comp, v);
    pl[e] = sum;
    cpl[e] = comp;
  } else {
    pl[e] += v;
  }
}

// Workgroups are dealt to the 8 XCDs round robin in dispatch order, and each
// XCD has its own L2.  A channel group's rows are often less than a 128-byte
// line, so neighbouring groups share lines: renumber the units so that
// consecutive units (neighbouring channel groups) run on the same XCD one
// after another and meet the line in its L2.
constexpr int kXcds = 8;
__device__ __forceinline__ long long xcd_swizzle(long long u, long long total) {
  const long long per = total / kXcds;  // units per XCD in the swizzled range
  if (u >= per * kXcds) return u;       // tail: unchanged
  return (u % kXcds) * per + u / kXcds;
}

// Segment of a multi-subband launch holding unit u (segments in order).
template <typename Seg>
__device__ __forceinline__ int find_seg(const Seg *segs, int nseg, long long u) {
  int s = 0;
  while (s + 1 < nseg && u >= segs[s + 1].unit0) ++s;
  return s;
}

}  // namespace xs
}  // namespace gxc
